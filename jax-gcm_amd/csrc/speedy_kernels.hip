// speedy_kernels.hip -- gfx950 kernels and the C ABI (include/speedy_abi.h) of the
// SPEEDY column physics.
//
// The eleven terms are column-local except for one grid-wide coupling: the
// shortwave cloud albedo is applied at every level of the set
//   S = { clip(icltop[c], 0, kx-1) : every column c of the call }
// (shortwave_radiation.py:63-70, an advanced-index scatter).  S is an OR of
// one bit per column, so a call needs a grid-wide reduction between the cloud
// top (end of phase A) and the shortwave (phase B).  Two paths:
//
//   fused (the grid fits on the GPU at once, e.g. T85 = 128 blocks):
//     one launch.  Right after the cloud top every block publishes its columns' OR
//     of level bits as one tagged word in its own slot (tag = the call's
//     generation), computes the S-independent work (longwave transmissivity,
//     longwave down, vertical diffusion), then polls only the slots of the blocks
//     covering its member until every tag is current.  A word that stays away
//     (its block is not running yet: other work holds the GPU) is formed by the
//     waiting block itself from the state, so no block depends on another one being
//     resident, and a plain launch is enough (a cooperative one took 20 us more).
//     Block 0 advances the generation once every block has published.  No
//     read-modify-write atomics in the exchange: contended same-address atomics cost
//     microseconds per call on this GPU.  Small batches run the same bodies.
//   two launches (larger grids, members narrower than a block, a given S, and
//     larger batches): a level-set kernel, a fixed number of blocks each covering a
//     contiguous chunk of columns, writes per-(chunk, member) ORs; the forward
//     kernel ORs the few chunks of its member, recomputes phase A and does
//     phase B.
//
// One thread per column; the column lives in registers.  Accesses are
// [field][level][column] with consecutive lanes on consecutive columns
// (coalesced 256-byte wave loads/stores).
#include <hip/hip_runtime.h>

#include <cstdio>
#include <algorithm>
#include <cstring>
#include <mutex>
#include <string>
#include <vector>

#include "speedy_adjoint.hpp"
#include "speedy_workspace.hpp"

namespace speedy {

static_assert(kParamParts == VJP_NPARAM && kBudParts == SPEEDY_NBUDGET + 1, "partials");

// Internal flag (above the public SPEEDY_FLAG_* bits): take the batch kernels' route
// even where the fused launch could run (speedy_fwd_noalloc).
constexpr uint32_t kFlagBatchRoute = 1u << 31;
// Polls (about 1 us each) before a block forms the words it misses itself.  In a
// GPU without other work the words are there after one or two; each word formed
// takes one wave about 10 us, so waiting out a short kernel of another stream is
// cheaper than replacing the blocks it holds up.
constexpr uint32_t kHelpAfter = 256;

struct Divisor {          // n / d for n < 2^32 by multiply-high + one correction step
  uint32_t d, m;          // m = floor(2^32 / d) (unused when d == 1)
};

struct KArgs {
  SpeedyFields f;
  SpeedyVertical v;
  SpeedyParams p;
  Uniforms<float> u;
  uint32_t ncol, ntot, nmember, nlat;
  uint32_t nblk;                     // blocks of kBlock columns
  uint32_t ls_blocks, chunk, jmax;   // two-kernel level-set pass: chunks of `chunk` columns
  Divisor dcol, dlat, dchunk;
  int32_t level_set;
  uint32_t flags, term_mask;
  uint32_t *gen, *err, *last_s, *partial;
  // fused forward + VJP only
  SpeedyAdjoint adj;
  uint32_t* arrived;                 // per member: blocks whose partials are out (zero between calls)
  uint32_t merged;                   // a fused call's members are summed in the launch (fused_sums)
  float* prm_part;                   // parameter-gradient partials (per block and member slot, or per column)
  double* bud_part;                  // float64 budget partials, kBudParts each (at block + member, or per column)
  void* desc;                        // a single call's argument block in its workspace
};

// ---------------------------------------------------------------- diagnostics
// Names follow Physics.data_struct_to_dict (physics_interface.py:157-194):
// "<struct>.<field>" and "<struct>.<field>.<channel>" for multi-channel fields.
static const char* kDiag2D[] = {
    "convection.iptop", "convection.cbmf", "convection.precnv", "condensation.precls",
    "shortwave_rad.icltop", "shortwave_rad.cloudc", "shortwave_rad.cloudstr", "shortwave_rad.qcloud",
    "shortwave_rad.gse", "shortwave_rad.rsds", "shortwave_rad.rsns", "shortwave_rad.ftop",
    "shortwave_rad.fsol", "shortwave_rad.ozupp", "shortwave_rad.ozone", "shortwave_rad.zenit",
    "shortwave_rad.stratz", "longwave_rad.ftop", "mod_radcon.albsfc", "mod_radcon.alb_l",
    "mod_radcon.alb_s", "mod_radcon.snowc", "mod_radcon.stratc.0", "mod_radcon.stratc.1",
    "mod_radcon.flux.0", "mod_radcon.flux.1", "mod_radcon.flux.2", "mod_radcon.flux.3",
    "surface_flux.ustr.0", "surface_flux.ustr.1", "surface_flux.ustr.2",
    "surface_flux.vstr.0", "surface_flux.vstr.1", "surface_flux.vstr.2",
    "surface_flux.shf.0", "surface_flux.shf.1", "surface_flux.shf.2",
    "surface_flux.evap.0", "surface_flux.evap.1", "surface_flux.evap.2",
    "surface_flux.rlus.0", "surface_flux.rlus.1", "surface_flux.rlus.2",
    "surface_flux.rlds", "surface_flux.rlns", "surface_flux.hfluxn.0", "surface_flux.hfluxn.1",
    "surface_flux.tsfc", "surface_flux.tskin", "surface_flux.u0", "surface_flux.v0", "surface_flux.t0"};
constexpr int kN2D = sizeof(kDiag2D) / sizeof(kDiag2D[0]);
static const char* kDiag3D[] = {
    "humidity.qsat", "humidity.rh", "convection.se", "shortwave_rad.dfabs", "longwave_rad.dfabs",
    "mod_radcon.st4a.0", "mod_radcon.st4a.1", "mod_radcon.tau2.0", "mod_radcon.tau2.1",
    "mod_radcon.tau2.2", "mod_radcon.tau2.3"};
constexpr int kN3D = sizeof(kDiag3D) / sizeof(kDiag3D[0]);

constexpr int diag_rows(int kx) { return kN2D + kN3D * kx; }

// ---------------------------------------------------------------- device helpers
__device__ __forceinline__ uint32_t divq(uint32_t n, const Divisor& dv) {
  if (dv.d == 1u) return n;
  uint32_t q = __umulhi(n, dv.m);
  if (n - q * dv.d >= dv.d) q += 1u;
  return q;
}

// Field access through address-space-1 (global) pointers.  The batch kernels
// read their field pointers from a descriptor in memory, and the compiler emits
// flat instructions for generic pointers; a flat access also counts in the
// scalar-load counter, so every wait for a uniform's scalar load then waits for
// the column's outstanding loads and stores too.  The kernel-argument kernels
// get global instructions either way.
template <typename T>
__device__ __forceinline__ T gld(const T* p, size_t i) {
  return ((const __attribute__((address_space(1))) T*)p)[i];
}
template <typename T>
__device__ __forceinline__ void gst(T* p, size_t i, T v) {
  ((__attribute__((address_space(1))) T*)p)[i] = v;
}

template <int KX, bool EXTRA>
__device__ __forceinline__ void load_state(const KArgs& a, uint32_t m, uint32_t c, ColumnIn<float, KX>& col) {
  const size_t ncol = a.ncol;
  const size_t base3 = (size_t)m * KX * ncol + c;
#pragma unroll
  for (int k = 0; k < KX; ++k) {
    col.T[k] = gld(a.f.t, base3 + k * ncol);
    col.Q[k] = gld(a.f.q, base3 + k * ncol);
    col.PHI[k] = gld(a.f.phi, base3 + k * ncol);
  }
  if (EXTRA && (a.flags & SPEEDY_FLAG_VERIFY_STATE)) {
#pragma unroll
    for (int k = 0; k < KX; ++k) col.Q[k] = verify_q(col.Q[k]);
  }
  col.u1 = gld(a.f.u, base3 + (KX - 1) * ncol);
  col.v1 = gld(a.f.v, base3 + (KX - 1) * ncol);
  col.ps = gld(a.f.ps, (size_t)m * ncol + c);
  col.alb0 = gld(a.f.alb0, c);
  col.sice = gld(a.f.sice_am, c);
  col.snowc_am = gld(a.f.snowc_am, c);
  col.soilw = gld(a.f.soilw_am, c);
  col.stl = gld(a.f.stl_am, c);
  col.sst = gld(a.f.sst, c);
  col.fmask = gld(a.f.fmask, c);
  col.orog = gld(a.f.orog, c);
  col.phis0 = gld(a.f.phis0, c);
}

template <int KX>
__device__ __forceinline__ void load_zonal(const KArgs& a, uint32_t c, ColumnIn<float, KX>& col) {
  const uint32_t j = c - divq(c, a.dlat) * a.nlat;
  float z[6];
  zonal_column(a.u.zon, gld(a.f.sia, j), gld(a.f.coa, j), z);
  col.fsol = z[0]; col.ozupp = z[1]; col.ozone = z[2]; col.zenit = z[3]; col.stratz = z[4]; col.sqcoa = z[5];
}

// u and v tendencies come from the surface stress at the lowest level only
// (surface_flux.py:294-295); the zeros above it are stored at the start of the
// kernel, off the critical path.
template <int KX>
__device__ __forceinline__ void store_uv_zeros(const KArgs& a, uint32_t m, uint32_t c) {
  const size_t ncol = a.ncol;
  const size_t base3 = (size_t)m * KX * ncol + c;
#pragma unroll
  for (int k = 0; k < KX - 1; ++k) {
    gst(a.f.du, base3 + k * ncol, 0.0f);
    gst(a.f.dv, base3 + k * ncol, 0.0f);
  }
}

// Up to eight levels, the term-ordered tendency sums (speedy_physics.py:123-125)
// are formed as early as their terms exist, in the same order of float
// additions: convection and condensation right after phase A; the q tendency of
// every level but the lowest once vertical diffusion (its last term there) is
// known.  The phase-A and vertical-diffusion tendencies then die early instead of
// staying live across phases b1 and b2 (16 fewer registers in the forward, and
// no scratch at two waves per SIMD).  The sixteen-level kernels keep the sums at
// the stores.
template <int KX>
constexpr bool kEarlySums = KX <= 8;

template <int KX>
__device__ __forceinline__ void tend_after_a(uint32_t tm, const PhaseA<float, KX>& pa, float at[KX], float aq[KX]) {
  if constexpr (!kEarlySums<KX>) return;
#pragma unroll
  for (int k = 0; k < KX; ++k) {
    float t = 0.0f, q = 0.0f;
    if (tm & (1u << SPEEDY_TERM_CONVECTION)) { t = t + pa.tconv[k]; q = q + pa.qconv[k]; }
    if (tm & (1u << SPEEDY_TERM_CONDENSATION)) { t = t + pa.tlsc[k]; q = q + pa.qlsc[k]; }
    at[k] = t;
    aq[k] = q;
  }
}
template <int KX>
__device__ __forceinline__ void tend_after_b1(uint32_t tm, const PhaseB<float, KX>& pb, float aq[KX]) {
  if constexpr (!kEarlySums<KX>) return;
  if (tm & (1u << SPEEDY_TERM_VDIFF)) {
#pragma unroll
    for (int k = 0; k < KX - 1; ++k) aq[k] = aq[k] + pb.qvd[k];
  }
}

// The diagnostics' rows (order of kDiag2D, then kDiag3D), stored as soon as they are
// final, so that phase b2 runs beside the stores and their 90 values leave the registers:
// the batch kernel then fits two waves per SIMD at 7 and 8 levels.  With all 140 rows
// stored at the end T213 took 62.9 us a call, now 49.1; T85 x 16 levels 39.8, now 34.4; T85
// x 8 18.0, now 17.7.  The fused kernels store after the level-set gather, whose loads
// would wait for the stores (T85 0.75 us slower before it).
template <int KX>
__device__ __forceinline__ float* diag_column(const KArgs& a, uint32_t m, uint32_t c) {
  return a.f.diag + (size_t)m * diag_rows(KX) * a.ncol + c;
}
template <int KX>
__device__ __forceinline__ void store_diag_a(const KArgs& a, uint32_t m, uint32_t c, const ColumnIn<float, KX>& col,
                                             const PhaseA<float, KX>& pa) {
  float* dg = diag_column<KX>(a, m, c);
  auto W = [&](int row, float x) { gst(dg, (size_t)row * a.ncol, x); };
  W(0, (float)pa.iptop); W(1, pa.cbmf); W(2, pa.precnv); W(3, pa.precls);
  W(4, (float)pa.icltop); W(5, pa.cloudc); W(6, pa.clstr); W(7, pa.qcloud); W(8, pa.gse);
  W(12, col.fsol); W(13, col.ozupp); W(14, col.ozone); W(15, col.zenit); W(16, col.stratz);
#pragma unroll
  for (int k = 0; k < KX; ++k) {
    W(kN2D + k, pa.qsat[k]); W(kN2D + KX + k, pa.rh[k]); W(kN2D + 2 * KX + k, pa.se[k]);
  }
}
template <int KX>
__device__ __forceinline__ void store_diag_b1(const KArgs& a, uint32_t m, uint32_t c, const PhaseB<float, KX>& pb) {
  float* dg = diag_column<KX>(a, m, c);
  auto W = [&](int row, float x) { gst(dg, (size_t)row * a.ncol, x); };
  W(18, pb.albsfc); W(19, pb.alb_l); W(20, pb.alb_s); W(21, pb.snowc);
#pragma unroll
  for (int k = 0; k < KX; ++k) {
    W(kN2D + 5 * KX + k, pb.st4a0[k]); W(kN2D + 6 * KX + k, pb.st4a1[k]);
#pragma unroll
    for (int b = 0; b < 4; ++b) W(kN2D + (7 + b) * KX + k, pb.tauL[k][b]);
  }
}

// at, aq: the partial sums of tend_after_a / tend_after_b1.
template <int KX, bool DIAG, bool EXTRA, bool FUSED>
__device__ __forceinline__ void store_outputs(const KArgs& a, uint32_t m, uint32_t c,
                                              const ColumnIn<float, KX>& col, const PhaseA<float, KX>& pa,
                                              const PhaseB<float, KX>& pb, const float at[KX], const float aq[KX],
                                              double colsum[2]) {
  const bool budget = EXTRA && a.f.budget != nullptr;
  const double dpg = (double)col.ps * (double)(P0 / GRAV);   // p0 ps / g; times dhs_k: dp_k / g
  colsum[0] = 0.0;
  colsum[1] = 0.0;
  // term-ordered sum (speedy_physics.py:123-125)
  const uint32_t tm = a.term_mask;
  const size_t ncol = a.ncol;
  const size_t base3 = (size_t)m * KX * ncol + c;
  // verify: the unclamped q again (L2), all levels ahead of the stores: a load between
  // them waits for the store before it (T425 with verify 107.2 -> 100.4 us a call, 64
  // members of T31 x 16 levels 136.6 -> 128.3, T85 16.9 -> 16.2).  The batched diagnostics
  // at 7 and 8 levels have no registers left for it.
  const bool verify = EXTRA && (a.flags & SPEEDY_FLAG_VERIFY_TENDENCIES) != 0u;
  constexpr bool kAhead = !DIAG || FUSED || KX > 8;
  float q_raw[KX];
  if (verify && kAhead)
#pragma unroll
    for (int k = 0; k < KX; ++k) q_raw[k] = gld(a.f.q, base3 + k * ncol);
#pragma unroll
  for (int k = 0; k < KX; ++k) {
    float t = 0.0f, q = 0.0f, du = 0.0f, dv = 0.0f;
    if (kEarlySums<KX>) {
      t = at[k];
      q = aq[k];
    } else {
      if (tm & (1u << SPEEDY_TERM_CONVECTION)) { t = t + pa.tconv[k]; q = q + pa.qconv[k]; }
      if (tm & (1u << SPEEDY_TERM_CONDENSATION)) { t = t + pa.tlsc[k]; q = q + pa.qlsc[k]; }
    }
    if (tm & (1u << SPEEDY_TERM_SHORTWAVE)) t = t + pb.tsw[k];
    if (k == KX - 1 && (tm & (1u << SPEEDY_TERM_SURFACE))) {
      du = du + pb.du1; dv = dv + pb.dv1; t = t + pb.dts1; q = q + pb.dqs1;
    }
    if (tm & (1u << SPEEDY_TERM_LW_UP)) t = t + pb.tlw[k];
    if (tm & (1u << SPEEDY_TERM_VDIFF)) {
      t = t + pb.tvd[k];
      if (!kEarlySums<KX> || k == KX - 1) q = q + pb.qvd[k];   // early sums: the levels above took it already
    }
    if (verify) {
      bool lim;
      q = verify_dq(kAhead ? q_raw[k] : gld(a.f.q, base3 + k * ncol), q, a.u.dt_step, lim);
    }
    if (k == KX - 1) {   // the levels above were zeroed by store_uv_zeros
      gst(a.f.du, base3 + k * ncol, du);
      gst(a.f.dv, base3 + k * ncol, dv);
    }
    gst(a.f.dt, base3 + k * ncol, t);
    gst(a.f.dq, base3 + k * ncol, q);
    if (budget) {
      const double dp = (double)a.v.dhs[k] * dpg;
      colsum[0] += (double)CP * (double)t * dp;
      colsum[1] += (double)q * dp;
    }
  }
  if (DIAG) {
    float* dg = diag_column<KX>(a, m, c);
    auto W = [&](int row, float x) { gst(dg, (size_t)row * ncol, x); };
    W(9, pb.rsds); W(10, pb.rsns); W(11, pb.ftop_sw); W(17, pb.ftop_lw);
    W(22, pb.stratc0); W(23, pb.stratc1);
    for (int i = 0; i < 4; ++i) W(24 + i, pb.flux_out[i]);
    for (int i = 0; i < 3; ++i) {
      W(28 + i, pb.ustr[i]); W(31 + i, pb.vstr[i]); W(34 + i, pb.shf[i]); W(37 + i, pb.evap[i]); W(40 + i, pb.rlus[i]);
    }
    W(43, pb.rlds); W(44, pb.rlns); W(45, pb.hfluxn[0]); W(46, pb.hfluxn[1]);
    W(47, pb.tsfc); W(48, pb.tskin); W(49, pb.u0); W(50, pb.v0); W(51, pb.t0);
#pragma unroll
    for (int k = 0; k < KX; ++k) {
      W(kN2D + 3 * KX + k, pb.dfabs_sw[k]);
      W(kN2D + 4 * KX + k, pb.dfl[k]);
    }
  }
}

// ---------------------------------------------------------------- level set S
// OR over the 64 lanes of a wave (all active): six data-parallel-primitive ORs
// within the register file (quad swaps, half-row and row mirrors give every lane
// its row's OR; the row-15 and row-31 broadcasts fold rows into row 3), then lane
// 63 is read: no LDS round trip.
__device__ __forceinline__ uint32_t wave_or(uint32_t v) {
  v |= __builtin_amdgcn_update_dpp(0u, v, 0xB1, 0xF, 0xF, false);    // quad_perm [1,0,3,2]
  v |= __builtin_amdgcn_update_dpp(0u, v, 0x4E, 0xF, 0xF, false);    // quad_perm [2,3,0,1]
  v |= __builtin_amdgcn_update_dpp(0u, v, 0x141, 0xF, 0xF, false);   // row_half_mirror
  v |= __builtin_amdgcn_update_dpp(0u, v, 0x140, 0xF, 0xF, false);   // row_mirror
  v |= __builtin_amdgcn_update_dpp(0u, v, 0x142, 0xA, 0xF, false);   // row_bcast:15 into rows 1, 3
  v |= __builtin_amdgcn_update_dpp(0u, v, 0x143, 0xC, 0xF, false);   // row_bcast:31 into rows 2, 3
  return __builtin_amdgcn_readlane(v, 63);
}

__device__ __forceinline__ uint32_t clip_bit(int icl, int kx) {
  return 1u << (icl < 0 ? 0 : (icl > kx - 1 ? kx - 1 : icl));
}

// Level bits of member m over the columns of block b (cloud tops from the state),
// by one wave with all lanes active: lanes on columns outside the member or the
// grid take the member's last column.
template <int KX>
__device__ __forceinline__ uint32_t block_level_bits(const KArgs& a, uint32_t b, uint32_t m) {
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t last = m * a.ncol + a.ncol - 1u;
  uint32_t bits = 0u;
  for (uint32_t i = 0; i < (uint32_t)kBlock; i += 64u) {
    const uint32_t gid = b * kBlock + i + lane;
    const bool mine = gid >= m * a.ncol && gid <= last;
    const uint32_t c = sel(mine, gid, last) - m * a.ncol;
    const size_t base3 = (size_t)m * KX * a.ncol + c;
    ColumnIn<float, KX> col;
#pragma unroll
    for (int k = 1; k < KX; ++k) {
      col.T[k] = gld(a.f.t, base3 + k * (size_t)a.ncol);
      const float q = gld(a.f.q, base3 + k * (size_t)a.ncol);
      col.Q[k] = sel((a.flags & SPEEDY_FLAG_VERIFY_STATE) != 0u, verify_q(q), q);
      col.PHI[k] = gld(a.f.phi, base3 + k * (size_t)a.ncol);
    }
    col.ps = gld(a.f.ps, (size_t)m * a.ncol + c);
    bits |= clip_bit(cloud_top<float, KX>(col, a.p, a.v, a.u), KX);
  }
  return bits;   // the member's last column is one of its own: its bit belongs to S
}

// The single launch's tagged words (speedy_workspace.hpp), per block and member slot:
// level bits, and partials of the parameter gradients (kParamParts each).
__device__ __forceinline__ uint64_t* level_words(const KArgs& a) {
  return reinterpret_cast<uint64_t*>(reinterpret_cast<char*>(a.gen) + kHeaderBytes);
}
__device__ __forceinline__ uint64_t* param_words(const KArgs& a) {
  return reinterpret_cast<uint64_t*>(reinterpret_cast<char*>(a.gen) + kHeaderBytes + kWordBytes);
}

// The call's results are invalid (speedy_workspace_status).
__device__ __forceinline__ void set_error(const KArgs& a) {
  __hip_atomic_store(a.err, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Between two polls of a wait: about 4 us, in short ones nothing to speak of.
__device__ __forceinline__ void poll_pause(bool brief) {
  if (brief) __builtin_amdgcn_s_sleep(1);
  else __builtin_amdgcn_s_sleep(100);
}

// One poll of the published words of the blocks covering member m: the OR of their
// level bits, and whether any word is not of this call yet.  By one wave, all lanes
// active throughout: lanes past the last word read it again (OR is idempotent).
__device__ __forceinline__ uint32_t poll_words(const KArgs& a, uint32_t tag, uint32_t m, bool& missing) {
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t b0 = (m * a.ncol) / kBlock, b1 = (m * a.ncol + a.ncol - 1u) / kBlock;
  uint32_t acc = 0;
  int stale = 0;
  for (uint32_t bb = b0; bb <= b1; bb += 64u) {
    const uint32_t b = min(bb + lane, b1);
    const uint32_t j = m - divq(b * kBlock, a.dcol);
    const uint64_t w = __hip_atomic_load(&level_words(a)[2u * b + j], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    stale |= (uint32_t)(w >> 32) != tag;
    acc |= (uint32_t)w;
  }
  missing = __any(stale);
  return wave_or(acc);
}

// Fused path: member m's level set, by one wave.  Polls the published words; after
// kHelpAfter polls (at once with SPEEDY_FLAG_NO_WAIT) every word still missing is
// formed here instead.
template <int KX>
__device__ __forceinline__ uint32_t collect_fused(const KArgs& a, uint32_t tag, uint32_t m) {
  const uint32_t patience = (a.flags & SPEEDY_FLAG_NO_WAIT) ? 0u : kHelpAfter;
  for (uint32_t spins = 0; spins < patience; ++spins) {
    bool missing;
    const uint32_t acc = poll_words(a, tag, m, missing);
    if (!missing) return acc;
    __builtin_amdgcn_s_sleep(1);
  }
  const uint32_t b0 = (m * a.ncol) / kBlock, b1 = (m * a.ncol + a.ncol - 1u) / kBlock;
  uint32_t acc = 0u;
  for (uint32_t b = b0; b <= b1; ++b) {   // uniform: every lane reads the same word
    const uint32_t j = m - divq(b * kBlock, a.dcol);
    const uint64_t w = __hip_atomic_load(&level_words(a)[2u * b + j], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (__builtin_amdgcn_readfirstlane((uint32_t)(w >> 32)) == tag && patience != 0u)
      acc |= (uint32_t)w;
    else
      acc |= block_level_bits<KX>(a, b, m);
  }
  return wave_or(acc);
}

// Block 0: every member's S to last_s (speedy_read_level_sets), then the next
// generation, once every block of the call has published (and so read this one).
__device__ __forceinline__ void finish_generation(const KArgs& a, uint32_t gen, uint32_t tag) {
  uint32_t spins = 0;
  for (uint32_t m = 0; m < a.nmember; ++m) {
    bool missing;
    uint32_t v = poll_words(a, tag, m, missing);
    while (missing) {
      if (spins >= kSpinLimit) {
        set_error(a);
        break;
      }
      poll_pause(spins++ < kShortPolls);
      v = poll_words(a, tag, m, missing);
    }
    gst(a.last_s, m, v);
  }
  __hip_atomic_store(a.gen, next_generation(gen), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Two-kernel path: member m's word of level-set chunk b (levelset_batch_kernel output).
__device__ __forceinline__ uint32_t chunk_word(const KArgs& a, uint32_t b, uint32_t m) {
  return gld(a.partial, b * a.jmax + (m - divq(b * a.chunk, a.dcol)));
}

// Two-kernel path, member wider than a block: this thread's share of the OR over
// the chunks covering member m, kChunkLoads words per thread.  Indexes past the
// member's last chunk are clamped to it (OR is idempotent), so the loads carry
// no branches and issue together.  A member spans at most ls_blocks <= 512
// chunks (make_grid), within the kChunkLoads * kBlock = 1024 this reaches.
constexpr uint32_t kChunkLoads = 4;
__device__ __forceinline__ uint32_t chunk_share(const KArgs& a, uint32_t m) {
  const uint32_t b0 = divq(m * a.ncol, a.dchunk), b1 = divq(m * a.ncol + a.ncol - 1u, a.dchunk);
  uint32_t acc = 0u;
#pragma unroll
  for (uint32_t r = 0; r < kChunkLoads; ++r) acc |= chunk_word(a, min(b0 + threadIdx.x + r * kBlock, b1), m);
  return acc;
}

// ---------------------------------------------------------------- kernels
// Two-kernel path, launch 1: every column's cloud top, ORed per (chunk, member).
template <int KX>
__device__ __forceinline__ void levelset_body(const KArgs& a, uint32_t bid, uint32_t* s_or) {
  const uint32_t c_begin = bid * a.chunk;
  const uint32_t c_end = min(c_begin + a.chunk, a.ntot);
  const uint32_t m_first = divq(c_begin, a.dcol);
  const uint32_t nm = divq(c_end - 1u, a.dcol) - m_first + 1u;
  for (uint32_t i = threadIdx.x; i < nm; i += kBlock) s_or[i] = 0u;
  __syncthreads();
  // kLsCols columns per thread per pass: all their loads issue before the first
  // cloud top is computed (at two waves per SIMD one column's loads leave the
  // memory latency exposed).  Columns past the chunk load column c_begin's
  // words (in bounds) and are not ORed.
  constexpr uint32_t kLsCols = 4;
  const size_t ncol = a.ncol;
  for (uint32_t g0 = c_begin + threadIdx.x; g0 < c_end; g0 += kLsCols * kBlock) {
    ColumnIn<float, KX> col[kLsCols];
    uint32_t mcol[kLsCols];
#pragma unroll
    for (uint32_t u = 0; u < kLsCols; ++u) {
      const uint32_t gid = g0 + u * kBlock < c_end ? g0 + u * kBlock : c_begin;
      const uint32_t m = divq(gid, a.dcol);
      const uint32_t c = gid - m * a.ncol;
      const size_t base3 = (size_t)m * KX * ncol + c;
      mcol[u] = m;
#pragma unroll
      for (int k = 1; k < KX; ++k) {
        col[u].T[k] = gld(a.f.t, base3 + k * ncol);
        col[u].Q[k] = gld(a.f.q, base3 + k * ncol);
        col[u].PHI[k] = gld(a.f.phi, base3 + k * ncol);
      }
      col[u].ps = gld(a.f.ps, (size_t)m * ncol + c);
    }
#pragma unroll
    for (uint32_t u = 0; u < kLsCols; ++u) {
      if (a.flags & SPEEDY_FLAG_VERIFY_STATE) {
#pragma unroll
        for (int k = 1; k < KX; ++k) col[u].Q[k] = verify_q(col[u].Q[k]);
      }
      if (g0 + u * kBlock < c_end)
        atomicOr(&s_or[mcol[u] - m_first], clip_bit(cloud_top<float, KX>(col[u], a.p, a.v, a.u), KX));
    }
  }
  __syncthreads();
  for (uint32_t i = threadIdx.x; i < nm; i += kBlock) gst(a.partial, bid * a.jmax + i, s_or[i]);
}

// Where a block's columns lie and what it knows of its members' level sets.
// Threads past the last column take the last column and do all its work, its
// stores included (the same values to the same addresses), so no store needs a
// branch; only the block sums leave them out.
struct BlockPos {
  uint32_t gid, m, c;       // global column, member and column of this thread
  bool active, wide;        // wide: a member is at least a block, so a block spans at most two members
  uint32_t m_first, nm;     // the block's first member and how many it spans
  uint32_t wave;            // this wave's index in the block, as a scalar: branches on it keep all lanes on
  uint32_t gen, tag;        // fused: the generation word and its tag (call_tag)
  uint32_t lw0, lw1;        // two launches: this thread's share of the members' chunk words
};

// ---------------------------------------------------------------- VJP helpers
// One column's slice of an LDS array laid out [slot][thread] (conflict-free).
struct LdsStore {
  static constexpr bool kOn = true;
  float* base;
  int off = 0;
  __device__ __forceinline__ void put(int i, float x) { base[i * kBlock + off] = x; }
  __device__ __forceinline__ float get(int i) const { return base[i * kBlock + off]; }
  // The same slots, read only after `dep` is computed (the offset passes through
  // an empty asm that takes dep), so the reads are not hoisted above it.
  __device__ __forceinline__ LdsStore after(float dep) const {
    LdsStore t = *this;
    asm volatile("" : "+v"(t.off) : "v"(dep));
    return t;
  }
};

template <int KX>
__device__ __forceinline__ void load_cotangents(const KArgs& a, uint32_t m, uint32_t c, ColumnCt<float, KX>& ct) {
  const size_t ncol = a.ncol;
  const size_t base3 = (size_t)m * KX * ncol + c;
  ct.du1 = gld(a.adj.ct_du, base3 + (KX - 1) * ncol);
  ct.dv1 = gld(a.adj.ct_dv, base3 + (KX - 1) * ncol);
#pragma unroll
  for (int k = 0; k < KX; ++k) {
    ct.dt[k] = gld(a.adj.ct_dt, base3 + k * ncol);
    ct.dq[k] = gld(a.adj.ct_dq, base3 + k * ncol);
  }
}

template <int KX>
__device__ __forceinline__ void store_grads(const KArgs& a, uint32_t m, uint32_t c, const ColumnAdj<float, KX>& g) {
  const size_t ncol = a.ncol;
  const size_t base3 = (size_t)m * KX * ncol + c;
#pragma unroll
  for (int k = 0; k < KX; ++k) {
    gst(a.adj.g_u, base3 + k * ncol, k == KX - 1 ? g.u1 : 0.0f);
    gst(a.adj.g_v, base3 + k * ncol, k == KX - 1 ? g.v1 : 0.0f);
    gst(a.adj.g_t, base3 + k * ncol, g.T[k]);
    gst(a.adj.g_q, base3 + k * ncol, g.Q[k]);
  }
  gst(a.adj.g_ps, (size_t)m * ncol + c, g.ps);
}

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

// One DPP step of a float sum: x plus the value DPP control CTRL selects (lanes
// outside ROWS keep x).
template <int CTRL, int ROWS>
__device__ __forceinline__ float dpp_add(float x) {
  return x + __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL, ROWS, 0xF, false));
}

// Float sum over the 64 lanes of a wave (all active) in a fixed order, by the
// DPP steps of wave_or (every lane holds its row's sum after the row mirror; the
// row broadcasts add rows 0-2 into row 3); the total is read from lane 63.
__device__ __forceinline__ float wave_sum_dpp(float v) {
  v = dpp_add<0xB1, 0xF>(v);    // quad_perm [1,0,3,2]
  v = dpp_add<0x4E, 0xF>(v);    // quad_perm [2,3,0,1]
  v = dpp_add<0x141, 0xF>(v);   // row_half_mirror
  v = dpp_add<0x140, 0xF>(v);   // row_mirror
  v = dpp_add<0x142, 0xA>(v);   // row_bcast:15 into rows 1, 3
  v = dpp_add<0x143, 0xC>(v);   // row_bcast:31 into rows 2, 3
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 63));
}

// Parameter gradients of this block: a fixed-order tree sum per member slot
// (deterministic), written to prm_part[block][slot][5].  Members narrower than
// a block write per-column values instead (prm_part[column][5]).  TAGGED: tagged words
// (param_words), for the block that sums the member in the same launch.
template <bool TAGGED>
__device__ __forceinline__ void block_param_partials(const KArgs& a, uint32_t bid, const BlockPos& b,
                                                     const float prm[VJP_NPARAM]) {
  if (!TAGGED && a.ncol < (uint32_t)kBlock) {
    if (b.active)
#pragma unroll
      for (int i = 0; i < VJP_NPARAM; ++i) gst(a.prm_part, (size_t)b.gid * VJP_NPARAM + i, prm[i]);
    return;
  }
  __shared__ float s_red[kBlock / 64][2 * VJP_NPARAM];
  const uint32_t lane = threadIdx.x & 63u, slot = b.m - b.m_first;
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    if (j > 0 && b.nm == 1u) break;   // uniform
#pragma unroll
    for (int i = 0; i < VJP_NPARAM; ++i) {
      const float v = wave_sum((b.active && slot == (uint32_t)j) ? prm[i] : 0.0f);
      if (lane == 0) s_red[b.wave][j * VJP_NPARAM + i] = v;
    }
  }
  __syncthreads();
  if (threadIdx.x < b.nm * VJP_NPARAM) {
    float acc = s_red[0][threadIdx.x];
#pragma unroll
    for (int w = 1; w < kBlock / 64; ++w) acc = acc + s_red[w][threadIdx.x];
    const size_t at = (size_t)bid * 2 * VJP_NPARAM + threadIdx.x;
    if constexpr (TAGGED)
      __hip_atomic_store(param_words(a) + at, tagged_word(b.tag, __builtin_bit_cast(uint32_t, acc)), __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
    else
      gst(a.prm_part, at, acc);
  }
}

__device__ __forceinline__ double wave_sum_d(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

__device__ __forceinline__ double wave_max_d(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o, 64));
  return v;
}

// Float64 budget partials of this block per member slot: weighted sums, the largest
// column water residual, and the weight sum.  Block b's of member m are at place b + m
// (the next block of a member, and the next member of a block, are both one further on).
// Members narrower than a block write per-column values instead.
__device__ __forceinline__ void block_budget_partials(const KArgs& a, uint32_t bid, const BlockPos& b,
                                                      const double v[kBudParts]) {
  // (formed again: the scalar registers are short at the end of a kernel)
  const uint32_t m_first = divq(bid * kBlock, a.dcol), slot = b.m - m_first;
  if (a.ncol < (uint32_t)kBlock) {
    if (b.active)
#pragma unroll
      for (int i = 0; i < kBudParts; ++i) gst(a.bud_part, (size_t)b.gid * kBudParts + i, v[i]);
    return;
  }
  __shared__ double s_bud[kBlock / 64][2 * kBudParts];
  const uint32_t wave = threadIdx.x >> 6, lane = threadIdx.x & 63u;
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int i = 0; i < kBudParts; ++i) {
      const bool mine = b.active && slot == (uint32_t)j;
      const double x = i == 5 ? wave_max_d(mine ? v[i] : 0.0) : wave_sum_d(mine ? v[i] : 0.0);
      if (lane == 0) s_bud[wave][j * kBudParts + i] = x;
    }
  __syncthreads();
  const uint32_t nm = divq(min(bid * kBlock + kBlock, a.ntot) - 1u, a.dcol) - m_first + 1u;
  if (threadIdx.x < nm * kBudParts) {
    const bool is_max = (threadIdx.x % kBudParts) == 5;
    double acc = s_bud[0][threadIdx.x];
#pragma unroll
    for (int w = 1; w < kBlock / 64; ++w) acc = is_max ? fmax(acc, s_bud[w][threadIdx.x]) : acc + s_bud[w][threadIdx.x];
    gst(a.bud_part, (size_t)(bid + m_first) * kBudParts + threadIdx.x, acc);
  }
}

// The forward.  FUSED: single launch with the level-set exchange; otherwise S comes
// from the level-set kernel of the same call or batch.
// EXTRA: the optional verify steps and float64 budgets are compiled in (their
// flags and pointers are then read at run time); the plain forward omits them.
// The batched forward kernels up to eight levels keep the longwave
// transmissivities in LDS between longwave down and longwave up (4 KX floats a
// column, [slot][thread]) instead of recomputing them per level (T425: 153 fewer
// VALU instructions a wave, ~1 % faster).  The fused kernels recompute: at one
// wave per SIMD the dependent LDS reads in the longwave-up sweep cost more than
// the exponentials (T85 forward ~2 % slower with the store).  The sixteen-level
// kernels keep their tested code.
template <bool ON>
__device__ __forceinline__ auto tau_store(float* s) {
  if constexpr (ON)
    return LdsStore{s + threadIdx.x};
  else
    return NoTauStore{};
}

// The thread's position, and the loads the level set needs, issued first so that
// their round trip overlaps the state's: the generation word (fused), or the level-set
// chunk words (a member wider than a block: each thread ORs its share of the
// chunks of the block's members; narrower: the <= 2 chunks covering its own).
template <bool FUSED>
__device__ __forceinline__ BlockPos block_pos(const KArgs& a, uint32_t bid) {
  BlockPos b;
  b.gid = bid * kBlock + threadIdx.x;
  b.active = b.gid < a.ntot;
  const uint32_t g0 = b.gid < a.ntot ? b.gid : a.ntot - 1u;
  b.m = divq(g0, a.dcol);
  b.c = g0 - b.m * a.ncol;
  const uint32_t blk0 = bid * kBlock;
  b.m_first = divq(blk0, a.dcol);
  b.nm = divq(min(blk0 + kBlock, a.ntot) - 1u, a.dcol) - b.m_first + 1u;   // <= 2 when fused
  b.wide = a.ncol >= (uint32_t)kBlock;
  b.wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  b.gen = b.tag = b.lw0 = b.lw1 = 0u;
  const bool need_s = a.level_set < 0;
  if (FUSED && need_s) {
    b.gen = __hip_atomic_load(a.gen, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    b.tag = call_tag(b.gen);
  }
  if (!FUSED && need_s) {
    if (b.wide) {
      b.lw0 = chunk_share(a, b.m_first);
      if (b.nm > 1u) b.lw1 = chunk_share(a, b.m_first + 1u);
    } else {
      const uint32_t b0 = divq(b.m * a.ncol, a.dchunk), b1 = divq(b.m * a.ncol + a.ncol - 1u, a.dchunk);
      b.lw0 = chunk_word(a, b0, b.m) | chunk_word(a, b1, b.m);
    }
  }
  return b;
}

// Fused: publish this block's word(s) for the call's level set, a wave-level OR
// per member slot (a fused block spans at most two members), then one word per slot.
__device__ __forceinline__ void publish_level_bits(const KArgs& a, uint32_t bid, const BlockPos& b, int icltop, int kx) {
  __shared__ uint32_t s_wor[kBlock / 64][2];
  const uint32_t bit = b.active ? clip_bit(icltop, kx) : 0u;
  const uint32_t o0 = wave_or(b.m == b.m_first ? bit : 0u), o1 = wave_or(b.m != b.m_first ? bit : 0u);
  s_wor[threadIdx.x >> 6][0] = o0;   // the wave's value, from every lane
  s_wor[threadIdx.x >> 6][1] = o1;
  __syncthreads();
  if (b.wave == 0u) {
    for (uint32_t j = 0; j < b.nm; ++j) {
      uint32_t w = 0u;
#pragma unroll
      for (int i = 0; i < kBlock / 64; ++i) w |= s_wor[i][j];
      __hip_atomic_store(&level_words(a)[2u * bid + j], tagged_word(b.tag, w), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
}

// Counts the block in for its members' sums (by one wave): s_last[j] becomes whether it
// is the last of member m_first + j.
__device__ __forceinline__ void count_in(const KArgs& a, const BlockPos& b, uint32_t* s_last) {
  for (uint32_t j = 0; j < b.nm; ++j) {
    const uint32_t m = b.m_first + j;
    const uint32_t n = (m * a.ncol + a.ncol - 1u) / kBlock - (m * a.ncol) / kBlock + 1u;
    uint32_t before = 0u;
    if ((threadIdx.x & 63u) == 0u)
      before = __hip_atomic_fetch_add(&a.arrived[m], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    before = __builtin_amdgcn_readfirstlane(before);
    const bool last = before == n - 1u;
    if (last) __hip_atomic_store(&a.arrived[m], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (before >= n) set_error(a);   // more than there are: calls overlap on this workspace
    s_last[j] = last;
  }
}

// The level set of this thread's member: gathered from the published words
// (fused) or from the chunk words (two launches), or the call's own.
template <int KX, bool FUSED, bool SUMS = false>
__device__ __forceinline__ uint32_t gather_level_set(const KArgs& a, uint32_t bid, const BlockPos& b,
                                                     uint32_t* s_last = nullptr) {
  if (a.level_set >= 0) return (uint32_t)a.level_set;
  if (FUSED) {
    __shared__ uint32_t s_s[2];
    if (b.wave == 0u) {   // wave 0 gathers S for the block's member(s)
      for (uint32_t j = 0; j < b.nm; ++j) s_s[j] = collect_fused<KX>(a, b.tag, b.m_first + j);
    } else if (b.wave == 1u && bid == 0u) {
      finish_generation(a, b.gen, b.tag);   // no other block waits for this one here: it has published
    } else if (SUMS && b.wave == 2u && a.merged) {
      count_in(a, b, s_last);
    }
    __syncthreads();
    return s_s[b.m - b.m_first];
  }
  uint32_t S = b.lw0;
  if (b.wide) {   // the block's OR per member slot
    __shared__ uint32_t s_lw[kBlock / 64][2];
    const uint32_t o0 = wave_or(b.lw0), o1 = wave_or(b.lw1);
    s_lw[threadIdx.x >> 6][0] = o0;   // the wave's value, from every lane
    s_lw[threadIdx.x >> 6][1] = o1;
    __syncthreads();
    S = 0u;
#pragma unroll
    for (int i = 0; i < kBlock / 64; ++i) S |= s_lw[i][b.m - b.m_first];
  }
  // every member's S for speedy_read_level_sets: the same word from each of its columns
  gst(a.last_s, b.m, S);
  return S;
}

// The float64 column budgets of this block (a.f.budget is set; block-uniform).
template <int KX>
__device__ __forceinline__ void column_budgets(const KArgs& a, uint32_t bid, const BlockPos& b, const PhaseA<float, KX>& pa,
                                               const PhaseB<float, KX>& pb, const double colsum[2]) {
  const uint32_t j = b.c - divq(b.c, a.dlat) * a.nlat;
  const double w = (double)gld(a.f.coa, j);
  const double E = (double)pb.evap2, P = (double)pa.precnv + (double)pa.precls;
  const double res = colsum[1] - (E - P);
  const double v[kBudParts] = {w * colsum[0], w * colsum[1], w * E, w * P, w * res, fabs(res), w};
  block_budget_partials(a, bid, b, v);
}

// The argument block (the launch's own, or a descriptor) read again: what follows loads
// its uniforms anew (scalar loads) where the scalar registers could not hold them from
// kernel entry and would spill them lane by lane into vector registers.
__device__ __forceinline__ const KArgs& reread(const void* args) {
  typedef const __attribute__((address_space(4))) KArgs* ConstPtr;
  ConstPtr p = (ConstPtr)args;
  asm volatile("" : "+s"(p));
  return *(const KArgs*)p;
}
template <int KX, bool DIAG, bool FUSED, bool EXTRA>
__device__ __forceinline__ void fwd_body(const KArgs& a, uint32_t bid) {
  constexpr bool kTau = !FUSED && KX <= 8;
  __shared__ float s_tau[kTau ? 4 * KX * kBlock : 1];
  const auto ts = tau_store<kTau>(s_tau);
  const BlockPos b = block_pos<FUSED>(a, bid);
  ColumnIn<float, KX> col;
  load_state<KX, EXTRA>(a, b.m, b.c, col);
  load_zonal<KX>(a, b.c, col);   // S-independent; its loads travel with the state's
  store_uv_zeros<KX>(a, b.m, b.c);
  PhaseA<float, KX> pa;
  phase_a<float, KX>(col, a.p, a.v, a.u, pa);
  float tend_t[KX], tend_q[KX];
  tend_after_a<KX>(a.term_mask, pa, tend_t, tend_q);
  if (FUSED && a.level_set < 0) publish_level_bits(a, bid, b, pa.icltop, KX);
  if (DIAG && !FUSED) store_diag_a<KX>(a, b.m, b.c, col, pa);
  PhaseB<float, KX> pb;
  phase_b1<float, KX>(col, pa, a.p, a.v, a.u, pb, ts);
  if (DIAG && !FUSED) store_diag_b1<KX>(a, b.m, b.c, pb);
  tend_after_b1<KX>(a.term_mask, pb, tend_q);
  const uint32_t S = gather_level_set<KX, FUSED>(a, bid, b);
  // with every output compiled in, the uniforms of phase b2 and the stores are read
  // again (T85 with diagnostics and verify: 17.2 -> 16.2 us; the plain forward is
  // 0.4 us slower that way)
  if (DIAG && FUSED) {
    store_diag_a<KX>(a, b.m, b.c, col, pa);
    store_diag_b1<KX>(a, b.m, b.c, pb);
  }
  const KArgs& o = !(DIAG && EXTRA) ? a
                   : FUSED          ? reread((const void*)__builtin_amdgcn_kernarg_segment_ptr())
                   : KX <= 8        ? reread(&a)
                                    : a;
  phase_b2<float, KX, DIAG>(col, pa, S, o.p, o.v, o.u, o.flags, pb, ts);
  double colsum[2] = {0.0, 0.0};
  store_outputs<KX, DIAG, EXTRA, FUSED>(o, b.m, b.c, col, pa, pb, tend_t, tend_q, colsum);
  if (EXTRA && a.f.budget) column_budgets<KX>(o, bid, b, pa, pb, colsum);
}

// Per-member parameter gradients from the partials, one block per member, in a
// fixed order (deterministic).
__device__ __forceinline__ void budget_reduce_body(const KArgs& a, uint32_t m) {
  double acc[kBudParts];
#pragma unroll
  for (int i = 0; i < kBudParts; ++i) acc[i] = 0.0;
  // (unrolled: several iterations' loads in flight; the order of the sums is the loop's)
  if (a.ncol >= (uint32_t)kBlock) {
    const uint32_t b0 = (m * a.ncol) / kBlock, b1 = (m * a.ncol + a.ncol - 1u) / kBlock;
#pragma unroll 4
    for (uint32_t b = b0 + threadIdx.x; b <= b1; b += kBlock)
#pragma unroll
      for (int i = 0; i < kBudParts; ++i) {
        const double x = gld(a.bud_part, (size_t)(b + m) * kBudParts + i);
        acc[i] = i == 5 ? fmax(acc[i], x) : acc[i] + x;
      }
  } else {
#pragma unroll 4
    for (uint32_t cc = threadIdx.x; cc < a.ncol; cc += kBlock)
#pragma unroll
      for (int i = 0; i < kBudParts; ++i) {
        const double x = gld(a.bud_part, ((size_t)m * a.ncol + cc) * kBudParts + i);
        acc[i] = i == 5 ? fmax(acc[i], x) : acc[i] + x;
      }
  }
  __shared__ double s_red[kBlock / 64][kBudParts];
  const uint32_t wave = threadIdx.x >> 6, lane = threadIdx.x & 63u;
#pragma unroll
  for (int i = 0; i < kBudParts; ++i) {
    const double v = i == 5 ? wave_max_d(acc[i]) : wave_sum_d(acc[i]);
    if (lane == 0) s_red[wave][i] = v;
  }
  __syncthreads();
  if (threadIdx.x < kBudParts) {
    const bool is_max = threadIdx.x == 5;
    double t = s_red[0][threadIdx.x];
#pragma unroll
    for (int w = 1; w < kBlock / 64; ++w) t = is_max ? fmax(t, s_red[w][threadIdx.x]) : t + s_red[w][threadIdx.x];
    s_red[0][threadIdx.x] = t;
  }
  __syncthreads();
  if (threadIdx.x < SPEEDY_NBUDGET) {
    const double wsum = s_red[0][SPEEDY_NBUDGET];
    const double t = s_red[0][threadIdx.x];
    gst(a.f.budget, (size_t)m * SPEEDY_NBUDGET + threadIdx.x, threadIdx.x == 5 ? t : t / wsum);
  }
}

// A block's partials of the parameter gradients, once they are of this call; NaN, and the
// error word set, if they do not come.
__device__ __forceinline__ void tagged_partials(const KArgs& a, size_t at, uint32_t tag, uint32_t& left,
                                                float x[VJP_NPARAM]) {
  uint64_t w[VJP_NPARAM];
  const bool here = await_words(
      tag, left,
      [&](int i) { return __hip_atomic_load(param_words(a) + at + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); },
      [](bool brief) { poll_pause(brief); }, w);
  if (!here) set_error(a);
#pragma unroll
  for (int i = 0; i < VJP_NPARAM; ++i) x[i] = here ? __builtin_bit_cast(float, (uint32_t)w[i]) : __builtin_nanf("");
}

template <bool TAGGED>
__device__ __forceinline__ void param_reduce_body(const KArgs& a, uint32_t m, uint32_t tag) {
  float acc[VJP_NPARAM];
#pragma unroll
  for (int i = 0; i < VJP_NPARAM; ++i) acc[i] = 0.0f;
  if constexpr (TAGGED) {
    uint32_t left = kSpinLimit;
    const uint32_t b0 = (m * a.ncol) / kBlock, b1 = (m * a.ncol + a.ncol - 1u) / kBlock;
#pragma unroll 1
    for (uint32_t b = b0 + threadIdx.x; b <= b1; b += kBlock) {   // twice at most (kFusedBlocks)
      const uint32_t j = m - divq(b * kBlock, a.dcol);
      float x[VJP_NPARAM];
      tagged_partials(a, ((size_t)b * 2 + j) * VJP_NPARAM, tag, left, x);
#pragma unroll
      for (int i = 0; i < VJP_NPARAM; ++i) acc[i] += x[i];
    }
  } else if (a.ncol >= (uint32_t)kBlock) {
    // (unrolled: several iterations' loads in flight; the order of the sums is the loop's)
    const uint32_t b0 = (m * a.ncol) / kBlock, b1 = (m * a.ncol + a.ncol - 1u) / kBlock;
#pragma unroll 4
    for (uint32_t b = b0 + threadIdx.x; b <= b1; b += kBlock) {
      const uint32_t j = m - divq(b * kBlock, a.dcol);
#pragma unroll
      for (int i = 0; i < VJP_NPARAM; ++i) acc[i] += gld(a.prm_part, ((size_t)b * 2 + j) * VJP_NPARAM + i);
    }
  } else {
#pragma unroll 4
    for (uint32_t cc = threadIdx.x; cc < a.ncol; cc += kBlock)
#pragma unroll
      for (int i = 0; i < VJP_NPARAM; ++i) acc[i] += gld(a.prm_part, ((size_t)m * a.ncol + cc) * VJP_NPARAM + i);
  }
  __shared__ float s_red[kBlock / 64][VJP_NPARAM];
  const uint32_t wave = threadIdx.x >> 6, lane = threadIdx.x & 63u;
#pragma unroll
  for (int i = 0; i < VJP_NPARAM; ++i) {
    const float v = wave_sum_dpp(acc[i]);
    if (lane == 0) s_red[wave][i] = v;
  }
  __syncthreads();
  if (threadIdx.x < VJP_NPARAM) {
    float t = s_red[0][threadIdx.x];
#pragma unroll
    for (int w = 1; w < kBlock / 64; ++w) t = t + s_red[w][threadIdx.x];
    gst(a.adj.g_params, (size_t)m * VJP_NPARAM + threadIdx.x, t);
  }
}

// Per-member sums of a call: parameter gradients (VJP) and float64 budgets.
__device__ __forceinline__ void member_reduce_body(const KArgs& a, uint32_t m) {
  if (a.adj.g_params) param_reduce_body<false>(a, m, 0u);
  if (a.f.budget) {
    __syncthreads();
    budget_reduce_body(a, m);
  }
}

// Fused forward + VJP: the block's partials, and the sums of the members that it was the
// last to be counted in for, in the order of member_reduce_body.  The count is taken
// while the block gathers the level set, so nobody waits for it; the blocks counted
// before are all running, and their partials carry the call's tag, so this one reads a
// block's words again until they have come: no fence between blocks (fences, which write
// the L2 caches back, cost more than the launch they save).  The five words of a block are
// read together; one after the other took T85 23.6 -> 25.2 us in graph replays.  A launch of its own took 3.9 us and
// a gap: 27.4 -> 26.0 us a call at T85 x 8 levels, 26.6 -> 25.3 at T42; counted at the end
// instead, T85 29.1 -> 28.8 us back to back, and 28.0 this way.
__device__ __forceinline__ void fused_sums(const KArgs& a, uint32_t bid, const BlockPos& b, const float prm[VJP_NPARAM],
                                           const uint32_t* s_last) {
  block_param_partials<true>(a, bid, b, prm);
  for (uint32_t j = 0; j < b.nm; ++j)
    if (__builtin_amdgcn_readfirstlane(s_last[j])) {
      param_reduce_body<true>(a, b.m_first + j, b.tag);
      __syncthreads();
    }
}

// Forward + VJP (all terms; the optional verify steps and budgets by run-time
// flags).  The forward's phase B and its reversal are interleaved
// (speedy_adjoint.hpp: the longwave's two sweeps; the surface fluxes and the
// shortwave reversed from their own tapes): nothing of phase B is computed twice
// but the up sweep's transmissivities, and the tendencies are the forward
// kernels' bit for bit.  The longwave tape lies in LDS, [slot][thread].
template <int KX, bool FUSED, bool STASH = !FUSED>
__device__ __forceinline__ void vjp_body(const KArgs& a, uint32_t bid) {
  // Values of phase A that phase B does not read wait in LDS (tvd, qsat and, up to
  // eight levels, rh above the top level) or are read again from memory (phi, dL/ddq), in
  // the kernels whose registers are short: the batched ones (two waves per SIMD at 7 and 8
  // levels, 79 floats a column with the tape: two blocks fill a CU's 160 KB).
  constexpr int kTape = vjp_tape_floats<KX>();
  constexpr bool kStash = STASH;
  constexpr int kStashRh = KX <= 8 ? KX - 1 : 0;
  __shared__ float s_tape[(kTape + (kStash ? 2 * KX + kStashRh : 0)) * kBlock];
  LdsStore tape{s_tape + threadIdx.x};
  const BlockPos b = block_pos<FUSED>(a, bid);
  const size_t ncol = a.ncol;
  const size_t base3 = (size_t)b.m * KX * ncol + b.c;
  ColumnIn<float, KX> col;
  load_state<KX, true>(a, b.m, b.c, col);
  load_zonal<KX>(a, b.c, col);
  store_uv_zeros<KX>(a, b.m, b.c);
  PhaseA<float, KX> pa;
  phase_a<float, KX>(col, a.p, a.v, a.u, pa);
  if (FUSED && a.level_set < 0) publish_level_bits(a, bid, b, pa.icltop, KX);
  // the term-ordered sums (speedy_physics.py:123-125), each term added as it exists
  float tend_t[KX], tend_q[KX];
#pragma unroll
  for (int k = 0; k < KX; ++k) {
    tend_t[k] = (0.0f + pa.tconv[k]) + pa.tlsc[k];
    tend_q[k] = (0.0f + pa.qconv[k]) + pa.qlsc[k];
  }
  ColumnCt<float, KX> ct;
  load_cotangents<KX>(a, b.m, b.c, ct);
  PhaseB<float, KX> pb;
  ColumnAdj<float, KX> g;
  VjpTapeB<float, KX> t;
  phase_b1_vjp<float, KX>(col, pa, a.p, a.v, a.u, ct, pb, g, t, tape);
  if constexpr (kStash) {
#pragma unroll
    for (int k = 0; k < KX; ++k) {
      tape.put(kTape + k, pb.tvd[k]);
      tape.put(kTape + KX + k, pa.qsat[k]);
      if (k > 0 && kStashRh > 0) tape.put(kTape + 2 * KX + k - 1, pa.rh[k]);
    }
  }
  __shared__ uint32_t s_last[2];
  const uint32_t S = gather_level_set<KX, FUSED, FUSED>(a, bid, b, s_last);
  phase_b2_taped<float, KX>(col, pa, S, a.p, a.v, a.u, a.flags, ct, pb, g, t);
  const bool budget = a.f.budget != nullptr;
  const double dpg = (double)col.ps * (double)(P0 / GRAV);   // p0 ps / g; times dhs_k: dp_k / g
  double colsum[2] = {0.0, 0.0};
  uint32_t limited = 0u;
#pragma unroll
  for (int k = 0; k < KX; ++k) {
    tend_t[k] = tend_t[k] + pb.tsw[k];
    float q = tend_q[k];
    if (k == KX - 1) { tend_t[k] = tend_t[k] + pb.dts1; q = q + pb.dqs1; }
    q = q + pb.qvd[k];
    if (a.flags & SPEEDY_FLAG_VERIFY_TENDENCIES) {
      bool lim;
      q = verify_dq(gld(a.f.q, base3 + k * ncol), q, a.u.dt_step, lim);   // the unclamped q (re-read, L2)
      limited |= (lim ? 1u : 0u) << k;
      ct.dq[k] = sel(lim, 0.0f, ct.dq[k]);   // its cotangent goes to the unclamped q alone (below)
    }
    gst(a.f.dq, base3 + k * ncol, q);
    if (budget) colsum[1] += (double)q * ((double)a.v.dhs[k] * dpg);
  }
  gst(a.f.du, base3 + (KX - 1) * ncol, 0.0f + pb.du1);
  gst(a.f.dv, base3 + (KX - 1) * ncol, 0.0f + pb.dv1);
  phase_b2_vjp<float, KX>(col, pa, S, a.p, a.v, a.u, ct, pb, g, t, tape);
  if constexpr (kStash) {
    uint32_t zero = 0u;   // an offset known only once the longwave is reversed: the reads below stay below
    asm volatile("" : "+v"(zero) : "v"(g.T[0]));
    const LdsStore st = tape.after(g.T[0]);
#pragma unroll
    for (int k = 0; k < KX; ++k) {
      const size_t e = base3 + k * ncol + zero;
      col.PHI[k] = gld(a.f.phi, e);
      ct.dq[k] = sel(((limited >> k) & 1u) != 0u, 0.0f, gld(a.adj.ct_dq, e));
      pb.tvd[k] = st.get(kTape + k);
      pa.qsat[k] = st.get(kTape + KX + k);
      pa.rh[k] = (k > 0 && kStashRh > 0) ? st.get(kTape + 2 * KX + k - 1) : mdiv(col.Q[k], pa.qsat[k]);
      pa.se[k] = (float)CP * col.T[k] + col.PHI[k];
    }
  }
#pragma unroll
  for (int k = 0; k < KX; ++k) {
    const float tt = (tend_t[k] + pb.tlw[k]) + pb.tvd[k];
    gst(a.f.dt, base3 + k * ncol, tt);
    if (budget) colsum[0] += (double)CP * (double)tt * ((double)a.v.dhs[k] * dpg);
  }
  if (budget) column_budgets<KX>(a, bid, b, pa, pb, colsum);
  phase_a_adj<float, KX>(col, pa, a.p, a.v, a.u, ct, g);
  if (a.flags & SPEEDY_FLAG_VERIFY_STATE) {
#pragma unroll
    for (int k = 0; k < KX; ++k) g.Q[k] = verify_q_grad(gld(a.f.q, base3 + k * ncol), g.Q[k]);
  }
  if (a.flags & SPEEDY_FLAG_VERIFY_TENDENCIES) {   // verify_ct's g_qraw (the cotangent re-read, L2)
#pragma unroll
    for (int k = 0; k < KX; ++k)
      g.Q[k] += sel(((limited >> k) & 1u) != 0u, -gld(a.adj.ct_dq, base3 + k * ncol) / a.u.dt_step, 0.0f);
  }
  store_grads<KX>(a, b.m, b.c, g);
  if (FUSED && a.merged) {
    if constexpr (STASH)   // a descriptor: as it is (segment)
      fused_sums(a, bid, b, g.prm, s_last);
    else
      fused_sums(reread(&a), bid, b, g.prm, s_last);
  } else {
    block_param_partials<false>(a, bid, b, g.prm);
  }
}


__global__ __launch_bounds__(kBlock) void param_reduce_kernel(KArgs a) { member_reduce_body(a, blockIdx.x); }

template <int KX, bool DIAG, bool FUSED, bool VJP, bool EXTRA>
__global__ __launch_bounds__(kBlock) void fwd_kernel(KArgs a) {
  // The forward + VJP reads its arguments through a pointer to the argument segment:
  // as by-value arguments they are all loaded at entry, and the scalar registers spill
  // into vector-register lanes (9039 -> 7629 VALU instructions at 8 levels).  The
  // forward keeps by-value arguments: its loads at entry hide behind the state's.
  if constexpr (VJP)
    vjp_body<KX, FUSED>(*(const KArgs*)__builtin_amdgcn_kernarg_segment_ptr(), blockIdx.x);
  else
    fwd_body<KX, DIAG, FUSED, EXTRA>(a, blockIdx.x);
}

// ---------------------------------------------------------------- batches
// A batch descriptor holds one KArgs per segment and, per launch, a table of
// (segment << 20 | block-in-segment) words; every block reads its word once and
// then works exactly as in the single-call kernels.
// A single call that the fused launch cannot take goes through the same kernels with no
// table and its argument block by value, or, in the kernels that are short of registers
// (sixteen levels, forward + VJP), in the workspace, written by the level-set launch.
// (A launch of its own that wrote it and the tables cost 2.3 us and a gap.)
constexpr uint32_t kSegShift = 20, kSegLocalMask = (1u << kSegShift) - 1u;

template <int KX>
constexpr bool kByValue = KX <= 8;   // forward kernels

// The workgroup's segment, and its block in it.  By value: either source is read-only
// to the launch and read through address space 4, so that the fields are scalar loads
// and move freely (T425 x 8 levels forward 97.8 -> 93.5 us, with the launch saved).
// The descriptor alone, __restrict__ in the kernels' signatures: scalar loads next to
// their use; through address space 4 they all move up and spill (64 members of T31 x
// 16 levels forward 126.8 us against 118.2, T425 x 8 levels forward + VJP 278 against 217).
template <int KX>
__device__ __forceinline__ const KArgs& segment(const KArgs* segs, const uint32_t* table, uint32_t& bid) {
  const uint32_t e = table ? __builtin_amdgcn_readfirstlane(table[blockIdx.x]) : blockIdx.x;
  bid = e & kSegLocalMask;
  if constexpr (kByValue<KX>) {
    typedef const __attribute__((address_space(4))) KArgs* ConstPtr;
    ConstPtr p = table ? (ConstPtr)segs + (e >> kSegShift) : (ConstPtr)__builtin_amdgcn_kernarg_segment_ptr();
    return *(const KArgs*)p;
  } else {
    return segs[e >> kSegShift];
  }
}

// Copies a by-value argument block to memory, by one workgroup.
__device__ __forceinline__ void write_desc(KArgs* dst) {
  const auto* src = (const __attribute__((address_space(4))) uint32_t*)__builtin_amdgcn_kernarg_segment_ptr();
  for (uint32_t w = threadIdx.x; w < (uint32_t)(sizeof(KArgs) / 4); w += kBlock)
    gst(reinterpret_cast<uint32_t*>(dst), w, src[w]);
}
__global__ __launch_bounds__(kBlock) void desc_kernel(KArgs, KArgs* desc) { write_desc(desc); }

// desc: where a single call's argument block goes that the next launch reads from memory.
template <int KX>
__global__ __launch_bounds__(kBlock) void levelset_batch_kernel(KArgs, const KArgs* segs, const uint32_t* table,
                                                                KArgs* desc) {
  extern __shared__ uint32_t s_or[];
  if (desc && blockIdx.x == 0) write_desc(desc);
  uint32_t bid;
  const KArgs& a = segment<8>(segs, table, bid);   // by value at every level count
  levelset_body<KX>(a, bid, s_or);
}

// Forward-only segments of a batch: the forward without the adjoint's registers.
template <int KX>
__global__ __launch_bounds__(kBlock, KX <= 8 ? 2 : 1) void fwd_only_batch_kernel(KArgs,
                                                                                 const KArgs* __restrict__ segs,
                                                                                 const uint32_t* __restrict__ table) {
  uint32_t bid;
  const KArgs& a = segment<KX>(segs, table, bid);
  fwd_body<KX, false, false, true>(a, bid);
}

// Forward-only segments of a batch in which none needs the verify steps or the
// float64 budgets: the forward without that optional code (4 % faster at T425).
// Both forward-only batch kernels are built for two waves per SIMD at 7 and 8
// levels (at most 256 registers a lane, no scratch): the second wave covers the
// first one's stalls, 128 -> 86 us at T425 x 8 levels.
template <int KX>
__global__ __launch_bounds__(kBlock, KX <= 8 ? 2 : 1) void fwd_plain_batch_kernel(KArgs,
                                                                                  const KArgs* __restrict__ segs,
                                                                                  const uint32_t* __restrict__ table) {
  uint32_t bid;
  const KArgs& a = segment<KX>(segs, table, bid);
  fwd_body<KX, false, false, false>(a, bid);
}

// Forward-only segments that also write the PhysicsData diagnostics: single
// calls with diagnostics that the fused launch cannot take.  Two waves per SIMD as
// in the kernels above (T213 59.7 -> 49.1 us).
template <int KX>
__global__ __launch_bounds__(kBlock, KX <= 8 ? 2 : 1) void fwd_diag_batch_kernel(KArgs, const KArgs* __restrict__ segs,
                                                                const uint32_t* __restrict__ table) {
  uint32_t bid;
  const KArgs& a = segment<KX>(segs, table, bid);
  fwd_body<KX, true, false, true>(a, bid);
}

// Forward + VJP segments of a batch.  Bound by VALU issue.  Built for two waves per
// SIMD at 7 and 8 levels (at most 256 registers a lane; 56 B of scratch at 8 levels,
// none at 7; 80 KB of LDS a block), one at 16 (512 registers, 156 KB of LDS, 212 B
// of scratch).  T425 x 8 levels: 412 -> 195 us, and 64 members of T31 x 16 levels:
// 2710 -> 275 us, against reversing every term from a recompute of its own
// (speedy_adjoint.hpp).  The descriptor is __restrict__, so uniforms are scalar
// loads next to their use (vector loads without it: 310 us at T425).  The fused kernel
// keeps one wave per SIMD and no scratch.
template <int KX>
__global__ __launch_bounds__(kBlock, KX <= 8 ? 2 : 1) void fwd_batch_kernel(const KArgs* __restrict__ segs,
                                                                            const uint32_t* __restrict__ table) {
  const uint32_t e = table ? __builtin_amdgcn_readfirstlane(table[blockIdx.x]) : blockIdx.x;
  vjp_body<KX, false>(segs[e >> kSegShift], e & kSegLocalMask);
}

// Batches of 7 or 8 levels whose blocks are co-resident (at most 512 of them, two a CU):
// the single-launch bodies on every segment, so the level sets are gathered in the
// launch and forward and forward + VJP segments run side by side.  Bound by the latency
// of its longest block, an adjoint's.  Built for two waves per SIMD as fwd_batch_kernel
// is (a block a CU would hold T85 twice).  Six requests from T21 to T85 (346 blocks):
// 32.5 us against 6.4 + 13.3 + 26.7 us and two gaps in the launches below, 216 -> 200 us
// a burst; four of T85 (512 blocks) 178 -> 165, all forward 122 -> 119.  Beyond that the
// kernels below have the higher occupancy or the leaner forward.
template <int KX>
__global__ __launch_bounds__(kBlock, 2) void small_batch_kernel(const KArgs* __restrict__ segs,
                                                             const uint32_t* __restrict__ table) {
  const uint32_t e = __builtin_amdgcn_readfirstlane(table[blockIdx.x]);
  const KArgs& a = segs[e >> kSegShift];
  if (a.adj.g_t)
    vjp_body<KX, true, true>(a, e & kSegLocalMask);
  else
    fwd_body<KX, false, true, true>(a, e & kSegLocalMask);
}

__global__ __launch_bounds__(kBlock) void param_reduce_batch_kernel(const KArgs* __restrict__ segs,
                                                                    const uint32_t* __restrict__ table) {
  const uint32_t e = __builtin_amdgcn_readfirstlane(table[blockIdx.x]);
  member_reduce_body(segs[e >> kSegShift], e & kSegLocalMask);
}

// acc[e] += diag[e] / steps for e < n (the diagnostics' running mean): four
// elements per thread (16-byte loads and stores when both buffers allow), a
// grid-stride loop, and the scalar tail by the first threads.
__global__ __launch_bounds__(kBlock) void diag_accumulate_kernel(const float* __restrict__ d, float* __restrict__ acc,
                                                                 int64_t n, float steps, int vec) {
  const int64_t stride = (int64_t)gridDim.x * kBlock;
  const int64_t t0 = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  int64_t done = 0;
  if (vec) {
    const int64_t n4 = n / 4;
    const float4* d4 = reinterpret_cast<const float4*>(d);
    float4* a4 = reinterpret_cast<float4*>(acc);
    for (int64_t i = t0; i < n4; i += stride) {
      const float4 x = d4[i];
      float4 y = a4[i];
      y.x += x.x / steps; y.y += x.y / steps; y.z += x.z / steps; y.w += x.w / steps;
      a4[i] = y;
    }
    done = n4 * 4;
  }
  for (int64_t i = done + t0; i < n; i += stride) acc[i] += d[i] / steps;
}

__global__ void fill_zero_kernel(uint32_t* p, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0u;
}

// ---------------------------------------------------------------- host side
thread_local std::string g_last_error;

int fail(int code, const std::string& msg) {
  g_last_error = msg;
  return code;
}

// kernel timers
struct Timer {
  std::mutex mu;
  bool on = false;
  int cap = 0, used = 0;
  std::vector<hipEvent_t> ev;   // begin/end per slot
  std::vector<int> kind;
} g_timer;

int timer_begin(hipStream_t s, int kind) {
  std::lock_guard<std::mutex> lk(g_timer.mu);
  if (!g_timer.on || g_timer.used >= g_timer.cap) return -1;
  const int slot = g_timer.used++;
  g_timer.kind[slot] = kind;
  (void)hipEventRecord(g_timer.ev[2 * slot], s);
  return slot;
}

void timer_end(hipStream_t s, int slot) {
  if (slot < 0) return;
  std::lock_guard<std::mutex> lk(g_timer.mu);
  (void)hipEventRecord(g_timer.ev[2 * slot + 1], s);
}

constexpr uint32_t kMaxJ = 16384;   // LDS words of the level-set kernel's per-member ORs

Divisor make_divisor(uint32_t d) {
  Divisor dv;
  dv.d = d;
  dv.m = d > 1 ? (uint32_t)(((uint64_t)1 << 32) / d) : 0u;
  return dv;
}

int check_fields(const SpeedyFields* f) {
  const void* req[] = {f->u, f->v, f->t, f->q, f->phi, f->ps, f->alb0, f->sice_am, f->snowc_am,
                       f->soilw_am, f->stl_am, f->sst, f->fmask, f->orog, f->phis0, f->sia, f->coa,
                       f->du, f->dv, f->dt, f->dq};
  for (const void* p : req)
    if (!p) return fail(SPEEDY_ERR_ARG, "speedy: a required field pointer is NULL");
  return SPEEDY_OK;
}

int prepare(const SpeedyFields* fields, const SpeedyVertical* vert, const SpeedyParams* params,
            const SpeedyDate* date, int32_t nlon, int32_t nlat, int32_t nmember, uint32_t flags,
            uint32_t term_mask, int32_t level_set, void* workspace, size_t workspace_bytes, KArgs& a,
            size_t tag_bytes = kTagBytes) {
  if (!fields || !vert || !params || !date) return fail(SPEEDY_ERR_ARG, "speedy: NULL struct argument");
  if (nlon <= 0 || nlat <= 0 || nmember <= 0) return fail(SPEEDY_ERR_ARG, "speedy: nlon, nlat, nmember must be > 0");
  if (vert->kx != 7 && vert->kx != 8 && vert->kx != 16)
    return fail(SPEEDY_ERR_KX, "speedy: kx must be 7, 8 or 16 (got " + std::to_string(vert->kx) + ")");
  if (flags & ~(uint32_t)SPEEDY_FLAGS_ALL) return fail(SPEEDY_ERR_ARG, "speedy: unknown flag bits");
  if ((flags & SPEEDY_FLAG_VERIFY_TENDENCIES) && !(date->dt_seconds > 0.0f))
    return fail(SPEEDY_ERR_ARG, "speedy: VERIFY_TENDENCIES needs date->dt_seconds > 0");
  if (term_mask & ~(uint32_t)SPEEDY_TERMS_ALL) return fail(SPEEDY_ERR_ARG, "speedy: unknown term bits");
  if (level_set >= (1 << vert->kx)) return fail(SPEEDY_ERR_ARG, "speedy: level_set has bits beyond kx");
  if (int rc = check_fields(fields)) return rc;
  const int64_t ncol = (int64_t)nlon * nlat;
  const int64_t ntot = ncol * nmember;
  if (ntot >= ((int64_t)1 << 31) - kBlock) return fail(SPEEDY_ERR_CAPACITY, "speedy: more than 2^31 columns per call");
  const Grid gr = make_grid(nlon, nlat, nmember);
  if (gr.jmax > kMaxJ) return fail(SPEEDY_ERR_CAPACITY, "speedy: too many members per column chunk");
  if (gr.ls_blocks > kChunkLoads * kBlock)   // chunk_share's reach (make_grid keeps it <= 512)
    return fail(SPEEDY_ERR_CAPACITY, "speedy: too many level-set chunks");
  const WsLayout L = ws_layout(gr, nmember, sizeof(KArgs), tag_bytes);
  if (!workspace) return fail(SPEEDY_ERR_WORKSPACE, "speedy: workspace is NULL");
  if (workspace_bytes < L.total)
    return fail(SPEEDY_ERR_WORKSPACE, "speedy: workspace too small (need " + std::to_string(L.total) + " bytes)");
  std::memset(&a, 0, sizeof(a));
  a.f = *fields;
  a.v = *vert;
  a.p = *params;
  make_uniforms(*params, *vert, *date, a.u);
  a.ncol = gr.ncol; a.ntot = gr.ntot; a.nmember = (uint32_t)nmember; a.nlat = (uint32_t)nlat;
  a.nblk = gr.nblk; a.ls_blocks = gr.ls_blocks; a.chunk = gr.chunk; a.jmax = gr.jmax;
  a.dcol = make_divisor(gr.ncol);
  a.dlat = make_divisor((uint32_t)nlat);
  a.dchunk = make_divisor(gr.chunk);
  a.level_set = level_set;
  a.flags = flags;
  a.term_mask = term_mask;
  char* w = static_cast<char*>(workspace);
  a.gen = reinterpret_cast<uint32_t*>(w);
  a.err = a.gen + 1;
  a.last_s = reinterpret_cast<uint32_t*>(w + L.last_s);
  a.partial = reinterpret_cast<uint32_t*>(w + L.partial);
  a.desc = w + L.desc;
  a.arrived = a.gen + kArrivedWord;
  a.merged = level_set < 0 && gr.ncol >= (uint32_t)kBlock && gr.nblk <= kFusedBlocks &&
             a.nmember <= kMergedMembers && !fields->budget;
  a.prm_part = reinterpret_cast<float*>(w + L.prm);
  a.bud_part = reinterpret_cast<double*>(w + L.bud);
  return SPEEDY_OK;
}

// Make sure the device's per-thread stack limit covers the kernel's private
// segment (register spills of the adjoint kernels: up to ~4 KB per lane at 16
// levels; HIP's default limit is 1 KB).  Called once per kernel before its
// first launch; raises the limit only.
template <typename K>
hipError_t ensure_stack(K kernel) {
  hipFuncAttributes fa;
  hipError_t e = hipFuncGetAttributes(&fa, reinterpret_cast<const void*>(kernel));
  if (e != hipSuccess) return e;
  size_t cur = 0;
  e = hipDeviceGetLimit(&cur, hipLimitStackSize);
  if (e != hipSuccess) return e;
  if ((size_t)fa.localSizeBytes > cur) e = hipDeviceSetLimit(hipLimitStackSize, (size_t)fa.localSizeBytes);
  return e;
}

// The stack limit the batch kernels of one level count need.
template <int KX>
hipError_t batch_stack() {
  hipError_t e = ensure_stack(fwd_batch_kernel<KX>);
  if (e == hipSuccess) e = ensure_stack(fwd_only_batch_kernel<KX>);
  if (e == hipSuccess) e = ensure_stack(fwd_plain_batch_kernel<KX>);
  if (e == hipSuccess) e = ensure_stack(fwd_diag_batch_kernel<KX>);
  return e;
}

// Largest grid that is co-resident on the current device for a kernel, as far as the
// workspace has words for it.
template <typename K>
int64_t coresident_blocks(K kernel) {
  int dev = 0, ncu = 0, per_cu = 0;
  if (hipGetDevice(&dev) != hipSuccess) return 0;
  if (hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) return 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, kBlock, 0) != hipSuccess) return 0;
  return std::min<int64_t>((int64_t)per_cu * ncu, kFusedBlocks);
}

template <int KX>
int64_t small_batch_blocks() {
  return ensure_stack(small_batch_kernel<KX>) == hipSuccess ? coresident_blocks(small_batch_kernel<KX>) : 0;
}

// One-time set-up of a kernel family: the stack limit its kernels need and the
// co-resident grid of its fused kernel.  A function-local static, so the first
// calls from several threads initialise it once (one GPU per process in this
// library's deployments).
struct LaunchInit {
  hipError_t err;
  int64_t cap;
};

template <int KX, bool DIAG, bool VJP, bool EXTRA>
int launch_fwd(const KArgs& a, hipStream_t s) {
  static const LaunchInit init = [] {
    hipError_t se = ensure_stack(fwd_kernel<KX, DIAG, true, VJP, EXTRA>);
    if (se == hipSuccess)
      se = VJP    ? ensure_stack(fwd_batch_kernel<KX>)
           : DIAG ? ensure_stack(fwd_diag_batch_kernel<KX>)
           : EXTRA ? ensure_stack(fwd_only_batch_kernel<KX>) : ensure_stack(fwd_plain_batch_kernel<KX>);
    return LaunchInit{se, se == hipSuccess ? coresident_blocks(fwd_kernel<KX, DIAG, true, VJP, EXTRA>) : 0};
  }();
  if (init.err != hipSuccess)
    return fail(SPEEDY_ERR_HIP, std::string("speedy: stack limit: ") + hipGetErrorString(init.err));
  const int64_t cap = init.cap;
  // Sixteen-level forward + VJP calls always take the batch route, whose kernel
  // keeps phase A in LDS and spills less.
  const bool fused = a.level_set < 0 && (int64_t)a.nblk <= cap && a.ncol >= (uint32_t)kBlock && !(VJP && KX == 16) &&
                     !(a.flags & kFlagBatchRoute);
  const int kind = VJP ? 2 : 1;
  hipError_t e = hipSuccess;
  if (fused) {
    const int slot = timer_begin(s, kind);
    hipLaunchKernelGGL((fwd_kernel<KX, DIAG, true, VJP, EXTRA>), dim3(a.nblk), dim3(kBlock), 0, s, a);
    e = hipGetLastError();
    timer_end(s, slot);
  } else {
    // Grids the fused launch cannot take (beyond one co-resident launch, members
    // narrower than a workgroup, or a given level set): the batch kernels on this one
    // call.
    if (a.nblk > kSegLocalMask)
      return fail(SPEEDY_ERR_CAPACITY, "speedy: more than 2^20 workgroups (2^28 columns) in one call");
    KArgs* desc = VJP || !kByValue<KX> ? static_cast<KArgs*>(a.desc) : nullptr;
    const KArgs* segs = desc;
    const uint32_t* table = nullptr;
    if (a.level_set < 0) {
      const int slot = timer_begin(s, 0);
      hipLaunchKernelGGL(levelset_batch_kernel<KX>, dim3(a.ls_blocks), dim3(kBlock), a.jmax * sizeof(uint32_t), s, a,
                         segs, table, desc);
      timer_end(s, slot);
    } else if (desc) {
      hipLaunchKernelGGL(desc_kernel, dim3(1), dim3(kBlock), 0, s, a, desc);
    }
    const int slot = timer_begin(s, kind);
    if (VJP)
      hipLaunchKernelGGL(fwd_batch_kernel<KX>, dim3(a.nblk), dim3(kBlock), 0, s, segs, table);
    else if (DIAG)
      hipLaunchKernelGGL(fwd_diag_batch_kernel<KX>, dim3(a.nblk), dim3(kBlock), 0, s, a, segs, table);
    else if (EXTRA)
      hipLaunchKernelGGL(fwd_only_batch_kernel<KX>, dim3(a.nblk), dim3(kBlock), 0, s, a, segs, table);
    else
      hipLaunchKernelGGL(fwd_plain_batch_kernel<KX>, dim3(a.nblk), dim3(kBlock), 0, s, a, segs, table);
    e = hipGetLastError();
    timer_end(s, slot);
  }
  // Per-member sums in a second small kernel, where the launch has not taken them.
  if (e == hipSuccess && ((VJP && !(fused && a.merged)) || a.f.budget)) {
    const int slot = timer_begin(s, 3);
    hipLaunchKernelGGL(param_reduce_kernel, dim3(a.nmember), dim3(kBlock), 0, s, a);
    timer_end(s, slot);
    e = hipGetLastError();
  }
  if (e != hipSuccess) return fail(SPEEDY_ERR_HIP, std::string("speedy: launch failed: ") + hipGetErrorString(e));
  return SPEEDY_OK;
}

bool needs_extra(const KArgs& a) {
  return (a.flags & (SPEEDY_FLAG_VERIFY_STATE | SPEEDY_FLAG_VERIFY_TENDENCIES)) || a.f.budget != nullptr;
}

template <int KX>
int launch_fwd_kx(const KArgs& a, hipStream_t s) {
  if (needs_extra(a))
    return a.f.diag ? launch_fwd<KX, true, false, true>(a, s) : launch_fwd<KX, false, false, true>(a, s);
  return a.f.diag ? launch_fwd<KX, true, false, false>(a, s) : launch_fwd<KX, false, false, false>(a, s);
}

// The forward + VJP has one instantiation, with the optional verify / budget code
// (run-time flags).
template <int KX>
int launch_fwd_vjp_kx(const KArgs& a, hipStream_t s) {
  return launch_fwd<KX, false, true, true>(a, s);
}

struct BatchLayout {
  size_t blk, ls, red, total;
};

int batch_layout(const SpeedySegment* segs, int32_t nseg, BatchLayout& L) {
  size_t nb = 0, nl = 0, nr = 0;
  for (int32_t i = 0; i < nseg; ++i) {
    const SpeedySegment& sg = segs[i];
    if (sg.nlon <= 0 || sg.nlat <= 0 || sg.nmember <= 0 ||
        (int64_t)sg.nlon * sg.nlat * sg.nmember >= ((int64_t)1 << 31) - kBlock)
      return fail(SPEEDY_ERR_ARG, "speedy_fwd_batch: bad grid in segment " + std::to_string(i));
    const Grid g = make_grid(sg.nlon, sg.nlat, sg.nmember);
    if (g.nblk > kSegLocalMask || g.ls_blocks > kSegLocalMask)
      return fail(SPEEDY_ERR_CAPACITY, "speedy_fwd_batch: segment " + std::to_string(i) + " too large for a batch");
    nb += g.nblk;
    if (sg.level_set < 0) nl += g.ls_blocks;
    if (sg.adj.g_t || sg.fields.budget) nr += (size_t)sg.nmember;
  }
  if (nb > 0x7fffffffu) return fail(SPEEDY_ERR_CAPACITY, "speedy_fwd_batch: too many blocks");
  L.blk = align256(sizeof(KArgs) * (size_t)nseg);
  L.ls = L.blk + align256(sizeof(uint32_t) * nb);
  L.red = L.ls + align256(sizeof(uint32_t) * nl);
  L.total = L.red + align256(sizeof(uint32_t) * (nr ? nr : 1));
  return SPEEDY_OK;
}

}  // namespace speedy

using namespace speedy;

extern "C" {

int speedy_abi_version(void) { return SPEEDY_ABI_VERSION; }

size_t speedy_workspace_bytes(int32_t nlon, int32_t nlat, int32_t nmember) {
  if (nlon <= 0 || nlat <= 0 || nmember <= 0) return 0;
  if ((int64_t)nlon * nlat * nmember >= ((int64_t)1 << 31) - kBlock) return 0;
  return ws_layout(make_grid(nlon, nlat, nmember), nmember, sizeof(KArgs)).total;
}

int speedy_workspace_init(void* workspace, size_t workspace_bytes, void* stream) {
  if (!workspace || workspace_bytes < 256) return fail(SPEEDY_ERR_WORKSPACE, "speedy: bad workspace");
  const int64_t n = (int64_t)(workspace_bytes / 4);
  hipLaunchKernelGGL(fill_zero_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0,
                     (hipStream_t)stream, (uint32_t*)workspace, n);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(SPEEDY_ERR_HIP, std::string("speedy: fill failed: ") + hipGetErrorString(e));
  return SPEEDY_OK;
}

int speedy_workspace_status(void* workspace, size_t workspace_bytes, uint32_t* status, void* stream) {
  if (!workspace || workspace_bytes < 256 || !status) return fail(SPEEDY_ERR_ARG, "speedy: bad arguments");
  uint32_t* err = static_cast<uint32_t*>(workspace) + 1;   // word 1: KArgs::err
  hipError_t e = hipMemcpyAsync(status, err, sizeof(uint32_t), hipMemcpyDeviceToHost, (hipStream_t)stream);
  if (e == hipSuccess) e = hipStreamSynchronize((hipStream_t)stream);
  if (e == hipSuccess && *status) {
    // a failed wait leaves late blocks' level-set words and the generation out of
    // step: the whole workspace starts again from zero
    const int64_t n = (int64_t)(workspace_bytes / 4);
    hipLaunchKernelGGL(fill_zero_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, (hipStream_t)stream,
                       static_cast<uint32_t*>(workspace), n);
    e = hipGetLastError();
  }
  if (e != hipSuccess) return fail(SPEEDY_ERR_HIP, std::string("speedy: status read failed: ") + hipGetErrorString(e));
  return SPEEDY_OK;
}

int speedy_diag_rows(int32_t kx) {
  if (kx != 7 && kx != 8 && kx != 16) return fail(-SPEEDY_ERR_KX, "speedy: kx must be 7, 8 or 16");
  return diag_rows(kx);
}

int speedy_diag_names(int32_t kx, char* buf, size_t buf_len) {
  if (kx != 7 && kx != 8 && kx != 16) return fail(SPEEDY_ERR_KX, "speedy: kx must be 7, 8 or 16");
  std::string s;
  for (int i = 0; i < kN2D; ++i) { if (!s.empty()) s += ","; s += kDiag2D[i]; }
  for (int i = 0; i < kN3D; ++i) { s += ","; s += kDiag3D[i]; s += "[]"; }
  if (!buf || buf_len < s.size() + 1) return fail(SPEEDY_ERR_ARG, "speedy: name buffer too small");
  std::memcpy(buf, s.c_str(), s.size() + 1);
  return SPEEDY_OK;
}

int speedy_fwd(const SpeedyFields* fields, const SpeedyVertical* vert, const SpeedyParams* params,
               const SpeedyDate* date, int32_t nlon, int32_t nlat, int32_t nmember, uint32_t flags,
               uint32_t term_mask, int32_t level_set, void* workspace, size_t workspace_bytes,
               void* stream) {
  KArgs a;
  if (int rc = prepare(fields, vert, params, date, nlon, nlat, nmember, flags, term_mask, level_set,
                       workspace, workspace_bytes, a))
    return rc;
  g_last_error.clear();
  hipStream_t s = (hipStream_t)stream;
  switch (vert->kx) {
    case 7: return launch_fwd_kx<7>(a, s);
    case 8: return launch_fwd_kx<8>(a, s);
    default: return launch_fwd_kx<16>(a, s);
  }
}

int speedy_fwd_vjp(const SpeedyFields* fields, const SpeedyAdjoint* adj, const SpeedyVertical* vert,
                   const SpeedyParams* params, const SpeedyDate* date, int32_t nlon, int32_t nlat, int32_t nmember,
                   uint32_t flags, int32_t level_set, void* workspace, size_t workspace_bytes, void* stream) {
  if (!adj) return fail(SPEEDY_ERR_ARG, "speedy: NULL adjoint struct");
  const void* req[] = {adj->ct_du, adj->ct_dv, adj->ct_dt, adj->ct_dq, adj->g_u, adj->g_v,
                       adj->g_t, adj->g_q, adj->g_ps, adj->g_params};
  for (const void* p : req)
    if (!p) return fail(SPEEDY_ERR_ARG, "speedy: a required adjoint pointer is NULL");
  if (fields && fields->diag) return fail(SPEEDY_ERR_ARG, "speedy: fwd_vjp writes no diagnostics (diag must be NULL)");
  KArgs a;
  if (int rc = prepare(fields, vert, params, date, nlon, nlat, nmember, flags, SPEEDY_TERMS_ALL, level_set,
                       workspace, workspace_bytes, a))
    return rc;
  a.adj = *adj;
  g_last_error.clear();
  hipStream_t s = (hipStream_t)stream;
  switch (vert->kx) {
    case 7: return launch_fwd_vjp_kx<7>(a, s);
    case 8: return launch_fwd_vjp_kx<8>(a, s);
    default: return launch_fwd_vjp_kx<16>(a, s);
  }
}

int speedy_fwd_batch(const SpeedySegment* segs, int32_t nseg, const SpeedyVertical* vert,
                     const SpeedyParams* params, void* desc, size_t desc_bytes, void* host_staging, void* stream) {
  if (!segs || nseg <= 0 || nseg > SPEEDY_BATCH_MAX_SEGMENTS || !vert || !params)
    return fail(SPEEDY_ERR_ARG, "speedy_fwd_batch: bad segment list");
  if (vert->kx != 7 && vert->kx != 8 && vert->kx != 16)
    return fail(SPEEDY_ERR_KX, "speedy_fwd_batch: kx must be 7, 8 or 16");
  BatchLayout L;
  if (int rc = batch_layout(segs, nseg, L)) return rc;
  if (!desc || !host_staging || desc_bytes < L.total)
    return fail(SPEEDY_ERR_WORKSPACE, "speedy_fwd_batch: descriptor buffers missing or too small (need " +
                                          std::to_string(L.total) + " bytes)");
  char* h = static_cast<char*>(host_staging);
  KArgs* ha = reinterpret_cast<KArgs*>(h);
  uint32_t* t_blk = reinterpret_cast<uint32_t*>(h + L.blk);
  uint32_t* t_ls = reinterpret_cast<uint32_t*>(h + L.ls);
  uint32_t* t_red = reinterpret_cast<uint32_t*>(h + L.red);
  // Co-resident, at 7 or 8 levels and with no member narrower than a workgroup: one
  // launch of small_batch_kernel (there both sides are measured).
  static const int64_t small_cap[2] = {small_batch_blocks<7>(), small_batch_blocks<8>()};
  int64_t blocks = 0;
  bool small = vert && (vert->kx == 7 || vert->kx == 8);
  for (int32_t i = 0; i < nseg; ++i) {
    const Grid g = make_grid(segs[i].nlon, segs[i].nlat, segs[i].nmember);
    blocks += g.nblk;
    small = small && g.ncol >= (uint32_t)kBlock;
  }
  small = small && blocks <= small_cap[vert->kx - 7];
  uint32_t nb = 0, nl = 0, nr = 0, jmax = 1;
  bool fwd_extra = false;   // a forward-only segment needs the verify steps or budgets
  std::vector<uint8_t> is_vjp((size_t)nseg, 0u);
  for (int32_t i = 0; i < nseg; ++i) {
    const SpeedySegment& sg = segs[i];
    if (sg.fields.diag) return fail(SPEEDY_ERR_ARG, "speedy_fwd_batch: segments write no diagnostics");
    const void* ap[] = {sg.adj.ct_du, sg.adj.ct_dv, sg.adj.ct_dt, sg.adj.ct_dq, sg.adj.g_u,
                        sg.adj.g_v, sg.adj.g_t, sg.adj.g_q, sg.adj.g_ps, sg.adj.g_params};
    int nset = 0;
    for (const void* q : ap) nset += q != nullptr;
    if (nset != 0 && nset != 10)
      return fail(SPEEDY_ERR_ARG, "speedy_fwd_batch: segment " + std::to_string(i) + " sets only some adjoint pointers");
    KArgs a;
    if (int rc = prepare(&sg.fields, vert, params, &sg.date, sg.nlon, sg.nlat, sg.nmember, sg.flags, SPEEDY_TERMS_ALL,
                         sg.level_set, sg.workspace, sg.workspace_bytes, a))
      return rc;
    a.adj = sg.adj;
    std::memcpy(&ha[i], &a, sizeof(KArgs));
    is_vjp[i] = nset != 0;
    if (!nset && needs_extra(a)) fwd_extra = true;
    if (a.level_set < 0 && !small) {
      for (uint32_t b = 0; b < a.ls_blocks; ++b) t_ls[nl++] = ((uint32_t)i << kSegShift) | b;
      jmax = std::max(jmax, a.jmax);
    }
    if ((nset && !(small && a.merged)) || sg.fields.budget)
      for (uint32_t m = 0; m < a.nmember; ++m) t_red[nr++] = ((uint32_t)i << kSegShift) | m;
  }
  // block table: the forward-only segments' blocks first, then the VJP segments'
  for (int pass = 0; pass < 2; ++pass)
    for (int32_t i = 0; i < nseg; ++i)
      if (is_vjp[i] == pass)
        for (uint32_t b = 0; b < ha[i].nblk; ++b) t_blk[nb++] = ((uint32_t)i << kSegShift) | b;
  uint32_t nbf = 0;
  for (int32_t i = 0; i < nseg; ++i)
    if (!is_vjp[i]) nbf += ha[i].nblk;
  uint32_t nbv = nb - nbf;
  g_last_error.clear();
  hipStream_t s = (hipStream_t)stream;
  hipError_t e = hipMemcpyAsync(desc, host_staging, L.total, hipMemcpyHostToDevice, s);
  if (e != hipSuccess) return fail(SPEEDY_ERR_HIP, std::string("speedy_fwd_batch: copy failed: ") + hipGetErrorString(e));
  const KArgs* d_args = static_cast<const KArgs*>(desc);
  const char* d = static_cast<const char*>(desc);
  const uint32_t* d_blk = reinterpret_cast<const uint32_t*>(d + L.blk);
  const uint32_t* d_ls = reinterpret_cast<const uint32_t*>(d + L.ls);
  const uint32_t* d_red = reinterpret_cast<const uint32_t*>(d + L.red);
  // The stack limit of each level count's batch kernels, raised once (a
  // function-local static: thread-safe); a failure fails every batch call.
  static const hipError_t stack_err[3] = {
      batch_stack<7>(), batch_stack<8>(), batch_stack<16>()};
  KArgs none;   // the kernels take a call's arguments by value or from the descriptor
  std::memset(&none, 0, sizeof(none));
  auto launch = [&](auto ls_kernel, auto fwd_only_b, auto fwd_plain_b, auto fwd_kernel_b, auto small_b,
                    int kxi) -> hipError_t {
    if (stack_err[kxi] != hipSuccess) return stack_err[kxi];
    if (small) {
      const int slot = timer_begin(s, nbv ? 2 : 1);
      hipLaunchKernelGGL(small_b, dim3(nb), dim3(kBlock), 0, s, d_args, d_blk);
      timer_end(s, slot);
      nbf = nbv = 0;
    }
    if (nl) {
      const int slot = timer_begin(s, 0);
      hipLaunchKernelGGL(ls_kernel, dim3(nl), dim3(kBlock), jmax * sizeof(uint32_t), s, none, d_args, d_ls,
                         (KArgs*)nullptr);
      timer_end(s, slot);
    }
    if (nbf) {
      const int slot = timer_begin(s, 1);
      if (fwd_extra)
        hipLaunchKernelGGL(fwd_only_b, dim3(nbf), dim3(kBlock), 0, s, none, d_args, d_blk);
      else
        hipLaunchKernelGGL(fwd_plain_b, dim3(nbf), dim3(kBlock), 0, s, none, d_args, d_blk);
      timer_end(s, slot);
    }
    if (nbv) {
      const int slot = timer_begin(s, 2);
      hipLaunchKernelGGL(fwd_kernel_b, dim3(nbv), dim3(kBlock), 0, s, d_args, d_blk + nbf);
      timer_end(s, slot);
    }
    if (nr) {
      const int slot2 = timer_begin(s, 3);
      hipLaunchKernelGGL(param_reduce_batch_kernel, dim3(nr), dim3(kBlock), 0, s, d_args, d_red);
      timer_end(s, slot2);
    }
    return hipSuccess;
  };
  hipError_t le;
  switch (vert->kx) {
    case 7:
      le = launch(levelset_batch_kernel<7>, fwd_only_batch_kernel<7>, fwd_plain_batch_kernel<7>, fwd_batch_kernel<7>,
                  small_batch_kernel<7>, 0);
      break;
    case 8:
      le = launch(levelset_batch_kernel<8>, fwd_only_batch_kernel<8>, fwd_plain_batch_kernel<8>, fwd_batch_kernel<8>,
                  small_batch_kernel<8>, 1);
      break;
    default:
      le = launch(levelset_batch_kernel<16>, fwd_only_batch_kernel<16>, fwd_plain_batch_kernel<16>,
                  fwd_batch_kernel<16>, fwd_batch_kernel<16>, 2);
      break;
  }
  if (le != hipSuccess) return fail(SPEEDY_ERR_HIP, std::string("speedy_fwd_batch: stack limit: ") + hipGetErrorString(le));
  e = hipGetLastError();
  if (e != hipSuccess) return fail(SPEEDY_ERR_HIP, std::string("speedy_fwd_batch: launch failed: ") + hipGetErrorString(e));
  return SPEEDY_OK;
}

size_t speedy_batch_desc_bytes(const SpeedySegment* segs, int32_t nseg) {
  if (!segs || nseg <= 0 || nseg > SPEEDY_BATCH_MAX_SEGMENTS) return 0;
  BatchLayout L;
  if (batch_layout(segs, nseg, L)) return 0;
  return L.total;
}

int speedy_read_level_sets(const void* workspace, size_t workspace_bytes, int32_t nmember, uint32_t* out,
                           void* stream) {
  if (!workspace || !out || nmember <= 0) return fail(SPEEDY_ERR_ARG, "speedy: bad arguments");
  const size_t at = kHeaderBytes + kTagBytes;   // WsLayout::last_s of every grid
  if (workspace_bytes < at + align256(sizeof(uint32_t) * (size_t)nmember))
    return fail(SPEEDY_ERR_WORKSPACE, "speedy: workspace too small");
  hipError_t e = hipMemcpyAsync(out, static_cast<const char*>(workspace) + at, sizeof(uint32_t) * nmember,
                                hipMemcpyDeviceToHost, (hipStream_t)stream);
  if (e == hipSuccess) e = hipStreamSynchronize((hipStream_t)stream);
  if (e != hipSuccess) return fail(SPEEDY_ERR_HIP, std::string("speedy: copy failed: ") + hipGetErrorString(e));
  return SPEEDY_OK;
}

int speedy_diag_accumulate(const float* diag, float* acc, int64_t n, float steps_to_average, void* stream) {
  if (n < 0 || !(steps_to_average > 0.0f)) return fail(SPEEDY_ERR_ARG, "speedy_diag_accumulate: bad n or steps");
  if (n == 0) return SPEEDY_OK;
  if (!diag || !acc) return fail(SPEEDY_ERR_ARG, "speedy_diag_accumulate: NULL buffer");
  const int vec = ((reinterpret_cast<uintptr_t>(diag) | reinterpret_cast<uintptr_t>(acc)) % 16u) == 0u;
  const int64_t work = vec ? (n + 3) / 4 : n;
  const int64_t blocks = std::min<int64_t>((work + kBlock - 1) / kBlock, 4096);
  hipLaunchKernelGGL(diag_accumulate_kernel, dim3((uint32_t)blocks), dim3(kBlock), 0, (hipStream_t)stream, diag, acc,
                     n, steps_to_average, vec);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(SPEEDY_ERR_HIP, std::string("speedy_diag_accumulate: ") + hipGetErrorString(e));
  return SPEEDY_OK;
}

int speedy_timer_enable(int32_t capacity) {
  if (capacity <= 0 || capacity > (1 << 20)) return fail(SPEEDY_ERR_ARG, "speedy_timer_enable: bad capacity");
  std::lock_guard<std::mutex> lk(g_timer.mu);
  for (hipEvent_t e : g_timer.ev) (void)hipEventDestroy(e);
  g_timer.ev.assign(2 * (size_t)capacity, nullptr);
  g_timer.kind.assign(capacity, 0);
  for (auto& e : g_timer.ev)
    if (hipEventCreate(&e) != hipSuccess) return fail(SPEEDY_ERR_HIP, "speedy_timer_enable: hipEventCreate failed");
  g_timer.cap = capacity;
  g_timer.used = 0;
  g_timer.on = true;
  return SPEEDY_OK;
}

int speedy_timer_disable(void) {
  std::lock_guard<std::mutex> lk(g_timer.mu);
  g_timer.on = false;
  return SPEEDY_OK;
}

int speedy_timer_read(float* ms_per_kind, int32_t* launches_per_kind, int32_t nkinds) {
  if (!ms_per_kind || !launches_per_kind || nkinds <= 0) return fail(SPEEDY_ERR_ARG, "speedy_timer_read: bad args");
  std::lock_guard<std::mutex> lk(g_timer.mu);
  for (int i = 0; i < nkinds; ++i) { ms_per_kind[i] = 0.0f; launches_per_kind[i] = 0; }
  for (int slot = 0; slot < g_timer.used; ++slot) {
    const int k = g_timer.kind[slot];
    float ms = 0.0f;
    if (hipEventSynchronize(g_timer.ev[2 * slot + 1]) != hipSuccess ||
        hipEventElapsedTime(&ms, g_timer.ev[2 * slot], g_timer.ev[2 * slot + 1]) != hipSuccess)
      return fail(SPEEDY_ERR_HIP, "speedy_timer_read: event query failed");
    if (k < nkinds) { ms_per_kind[k] += ms; launches_per_kind[k] += 1; }
  }
  g_timer.used = 0;
  return SPEEDY_OK;
}

const char* speedy_last_error(void) { return g_last_error.c_str(); }

}  // extern "C"

// ---------------------------------------------------------------- allocation-free forward
// speedy_fwd_noalloc: speedy_fwd with its workspace in this file-scope device
// array instead of a caller's buffer, for callers that cannot allocate.  Each GPU
// holds its own copy for the life of the process; its device address is looked
// up once per device (hipGetSymbolAddress) and only that address is passed to
// kernels.  Calls take the batch kernels' route, which has no tagged words and reads no
// word of the workspace that the same call has not written first (descriptor, chunk
// words, partials), so the contents left by an earlier call, of any grid, are
// never read and nothing needs clearing.  Calls that overlap on one GPU share
// the array and race.
namespace speedy {
constexpr size_t kNoAllocScratchBytes = (size_t)4 << 20;
__device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];

constexpr int kNoAllocMaxDevices = 64;
std::mutex g_noalloc_mu;
void* g_noalloc_ptr[kNoAllocMaxDevices] = {};
}  // namespace speedy

extern "C" size_t speedy_noalloc_max_bytes(void) { return kNoAllocScratchBytes; }

extern "C" int speedy_fwd_noalloc(const SpeedyFields* fields, const SpeedyVertical* vert, const SpeedyParams* params,
                                  const SpeedyDate* date, int32_t nlon, int32_t nlat, int32_t nmember, uint32_t flags,
                                  uint32_t term_mask, int32_t level_set, void* stream) {
  if (speedy_workspace_bytes(nlon, nlat, nmember) == 0) return fail(SPEEDY_ERR_ARG, "speedy_fwd_noalloc: bad grid");
  const size_t need = ws_layout(make_grid(nlon, nlat, nmember), nmember, sizeof(KArgs), 0).total;
  if (need > kNoAllocScratchBytes)
    return fail(SPEEDY_ERR_CAPACITY, "speedy_fwd_noalloc: the call needs " + std::to_string(need) +
                                         " bytes of workspace, above the " + std::to_string(kNoAllocScratchBytes) +
                                         "-byte static scratch; use speedy_fwd with a caller workspace");
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return fail(SPEEDY_ERR_HIP, std::string("speedy_fwd_noalloc: ") + hipGetErrorString(e));
  if (dev < 0 || dev >= kNoAllocMaxDevices) return fail(SPEEDY_ERR_CAPACITY, "speedy_fwd_noalloc: device index");
  void* ws = nullptr;
  {
    std::lock_guard<std::mutex> lk(g_noalloc_mu);
    if (!g_noalloc_ptr[dev]) {
      void* p = nullptr;
      e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
      if (e != hipSuccess || !p)
        return fail(SPEEDY_ERR_HIP, std::string("speedy_fwd_noalloc: scratch address: ") + hipGetErrorString(e));
      g_noalloc_ptr[dev] = p;
    }
    ws = g_noalloc_ptr[dev];
  }
  KArgs a;
  if (int rc = prepare(fields, vert, params, date, nlon, nlat, nmember, flags, term_mask, level_set, ws,
                       kNoAllocScratchBytes, a, 0))
    return rc;
  a.flags |= kFlagBatchRoute;
  g_last_error.clear();
  hipStream_t s = (hipStream_t)stream;
  switch (vert->kx) {
    case 7: return launch_fwd_kx<7>(a, s);
    case 8: return launch_fwd_kx<8>(a, s);
    default: return launch_fwd_kx<16>(a, s);
  }
}
