// Voxel-driven cone-beam backprojection for gfx950.
//
// Behaviour follows cone_bp of the reference (kernelkit/cuda/cone_bp.cu:
// 35-159, launched by kernelkit/kernels/cone_bp.py:292-302): for every voxel
// centre X and angle, r = 1/den(X), (u, v) = (numU(X), numV(X)) * r, the
// projection is sampled bilinearly at (u, v) with zero outside, and
// r^2 * sample is accumulated; the sum is scaled by the voxel volume.
//
// MI355X design:
// * one launch covers all angles (the reference launches per batch of 32
//   angles and read-modify-writes the volume each time); each voxel is
//   written once, or updated in place by the fused SIRT epilogue;
// * a thread owns K consecutive voxels along z in registers.  For a circular
//   orbit about z the column coordinate u and the weight 1/den do not depend
//   on z, so the reciprocal, u and its interpolation weights are computed
//   once per (x, y, angle) and shared by the K voxels; rows advance by a
//   constant step.  A detector tilted in its own plane keeps 1/den shared
//   (u and v both affine along the run); other geometries take the
//   general per-voxel path (a wave-uniform branch per angle);
// * projections are read from a zero-halo texture of (value, next-row)
//   float2 pairs (kk_internal.h): a sample is a clamp, ONE 16-byte load for
//   the four taps and three lerps, with no bounds tests (the
//   texture-address unit, not the ALU, limits a gather kernel);
// * lanes of a wavefront are a 16 x 4 (x, y) patch, which projects onto a
//   compact detector patch; on circular orbits workgroups go to the XCDs
//   in groups of 4 x 4 x 4 neighbouring tiles, whose detector patches
//   overlap, otherwise in runs of 16 tiles along x.
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "kk_internal.h"

namespace {

constexpr int kMaxFrames = 3;

struct BpArgs {
  const char* tex;   // projection texture (byte base)
  uint32_t tab_b;    // bytes per angle image ((rows+3) * (cols+3) * 8)
  uint32_t trb;      // bytes per texture row ((cols+3) * 8)
  int32_t nx, ny, nz, n_angles, rows, cols;
  float* out;
  int64_t vs0, vs1, vs2;  // output world strides
  float scale;
  int32_t mode;  // 0: out = b, 1: out += b, 2: SIRT update
  int32_t tiles_x, tiles_y, tiles_z;
  int32_t xcd_group;
  int32_t gx, gy, gz;  // tiles per workgroup group along x, y, z
  int64_t total_blocks;
  // mode 2: x <- clip(mask * (x - C * b)), mirrored into the FP textures
  const float* C;
  int64_t cs0, cs1, cs2;
  const float* mask;
  int64_t ms0, ms1, ms2;
  float lo, hi;
  int32_t clip_lo, clip_hi;
  float* xtex;
  int32_t n_frames;
  int64_t fr_origin[kMaxFrames], fr_s0[kMaxFrames], fr_s1[kMaxFrames],
      fr_s2[kMaxFrames], fr_dual[kMaxFrames];
};

// Bilinear value from the 16-byte tap record (p[r][c], p[r+1][c],
// p[r][c+1], p[r+1][c+1]): lerp along rows (fv), then columns (fu).
__device__ __forceinline__ float bilerp(kk_float4u t, float fu, float fv) {
  const float l0 = fmaf(fv, t.y - t.x, t.x);
  const float l1 = fmaf(fv, t.w - t.z, t.z);
  return fmaf(fu, l1 - l0, l0);
}

// 1/den from a float32 estimate and one float64 Newton step (relative
// error ~1e-14).
__device__ __forceinline__ double refine_rcp(double den, float rf) {
  const double r = static_cast<double>(rf);
  return fma(r, fma(-den, r, 1.0), r);
}

// Coordinate base + off (base an integer, off a small float) clamped into
// [0, hi] (the zero halo), split into element index and weight: the same
// result as clamping the float64 coordinate, then floor and fraction.
// The clamp is applied to off, into [lo, up] = [-base, hi - base] (integers,
// exact in float32 for |base|, hi < 2^24; the caller passes them
// converted), so at either bound the weight is 0 and the index 0 or hi.
__device__ __forceinline__ void split_clamped(float off, int32_t base,
                                              float lo, float up,
                                              int32_t& idx, float& frac) {
  const float o = __builtin_amdgcn_fmed3f(off, lo, up);
  const float fl = floorf(o);
  idx = base + static_cast<int32_t>(fl);
  frac = o - fl;
}

// split_clamped for a coordinate known to lie in [0, hi): no clamps, the
// same index and weight.
__device__ __forceinline__ void split_inside(float off, int32_t base,
                                             int32_t& idx, float& frac) {
  const float fl = floorf(off);
  idx = base + static_cast<int32_t>(fl);
  frac = off - fl;
}

// Whether base + [lo, hi_off] lies in [1, hi - 1]: a run of coordinates
// there never reaches split_clamped's clamps (one texel of margin covers
// the float32 evaluation of this test).
__device__ __forceinline__ bool run_inside(int32_t base, float lo,
                                           float hi_off, int32_t hi) {
  const float b = static_cast<float>(base);
  return b + lo >= 1.f && b + hi_off <= static_cast<float>(hi - 1);
}

// Tile (tx, ty, tz) of logical block id `bid`: groups of gx x gy x gz tiles
// (x fastest inside), groups ordered x -> y -> z (the group sides divide the
// tile counts; 1 x 1 x 1 is plain x -> y -> z order).
__device__ __forceinline__ bool bp_decode(const BpArgs& A, int64_t bid,
                                          int32_t& tx, int32_t& ty,
                                          int32_t& tz) {
  const int32_t gx = A.gx, gy = A.gy, gz = A.gz;
  const int64_t inner = bid % (gx * gy * gz);
  const int64_t outer = bid / (gx * gy * gz);
  const int32_t ngx = (A.tiles_x + gx - 1) / gx;
  const int32_t ngy = (A.tiles_y + gy - 1) / gy;
  tx = static_cast<int32_t>(outer % ngx) * gx +
       static_cast<int32_t>(inner % gx);
  const int64_t o2 = outer / ngx;
  ty = static_cast<int32_t>(o2 % ngy) * gy +
       static_cast<int32_t>((inner / gx) % gy);
  tz = static_cast<int32_t>(o2 / ngy) * gz +
       static_cast<int32_t>(inner / (gx * gy));
  return tx < A.tiles_x && ty < A.tiles_y && tz < A.tiles_z;
}

// Write the sum `acc` of voxel (ix, iy, iz) as the launch's mode says.
__device__ __forceinline__ void bp_store(const BpArgs& A, int32_t ix,
                                         int32_t iy, int32_t iz, float acc) {
  const int64_t o = ix * A.vs0 + iy * A.vs1 + iz * A.vs2;
  const float b = acc * A.scale;
  if (A.mode == 0) {
    A.out[o] = b;
  } else if (A.mode == 1) {
    A.out[o] += b;
  } else {
    float x = A.out[o] - A.C[ix * A.cs0 + iy * A.cs1 + iz * A.cs2] * b;
    if (A.mask) x *= A.mask[ix * A.ms0 + iy * A.ms1 + iz * A.ms2];
    if (A.clip_lo) x = fmaxf(x, A.lo);
    if (A.clip_hi) x = fminf(x, A.hi);
    A.out[o] = x;
    for (int f = 0; f < A.n_frames; ++f) {
      const int64_t q = A.fr_origin[f] + ix * A.fr_s0[f] +
                        iy * A.fr_s1[f] + iz * A.fr_s2[f];
      A.xtex[q] = x;
      A.xtex[q + A.fr_dual[f]] = x;
    }
  }
}

// One workgroup's tile (16 x 16 columns of K voxels) of logical block id
// `bid`.  TABLE_IN_MEMORY: the angle table pointer was read from a
// descriptor (batch kernel), so each record is copied through
// constant-memory (scalar) loads; a kernel-argument table is read in place.
template <int K, bool TABLE_IN_MEMORY>
__device__ __forceinline__ void bp_tile(const kk::BpAngle* __restrict__ tab,
                                        const BpArgs& A, int64_t bid) {
  int32_t tx, ty, tz;
  if (!bp_decode(A, bid, tx, ty, tz)) return;
  const int32_t ix = tx * 16 + int32_t(threadIdx.x & 15);
  const int32_t iy = ty * 16 + int32_t(threadIdx.x >> 4);
  const int32_t iz0 = tz * K;
  if (ix >= A.nx || iy >= A.ny) return;

  // voxel centres; the geometry is evaluated in float64 per (x, y, angle):
  // detector coordinates reach ~cols + 1 (up to ~1.5e3), where float32
  // would round them by ~1e-4 pixel.  Per voxel only small offsets from an
  // integer base are float32.
  const double X = static_cast<double>(ix) - 0.5 * A.nx + 0.5;
  const double Y = static_cast<double>(iy) - 0.5 * A.ny + 0.5;
  const double Z0 = static_cast<double>(iz0) - 0.5 * A.nz + 0.5;
  const int32_t rmax = A.rows + 1;
  const int32_t cmax = A.cols + 1;
  const uint32_t trb = A.trb;

  float acc[K];
#pragma unroll
  for (int k = 0; k < K; ++k) acc[k] = 0.f;

  const char* img = A.tex;
  for (int32_t a = 0; a < A.n_angles; ++a, img += A.tab_b) {
    kk::BpAngle rec;
    const kk::BpAngle& P =
        TABLE_IN_MEMORY ? (rec = kk_uniform_load(tab + a), rec) : tab[a];
    const double den = fma(Y, P.dy, fma(X, P.dx, P.dw));
    const double nu = fma(Y, P.nuy, fma(X, P.nux, P.nuw));
    const double nv = fma(Y, P.nvy, fma(X, P.nvx, P.nvw));
    if (P.fast == 2) {
      // 1/den and the weight do not depend on z; u and v are affine in z
      const float rf = __builtin_amdgcn_rcpf(static_cast<float>(den));
      const double r = refine_rcp(den, rf);
      const double u0 = fma(Z0, P.nuz, nu) * r;
      const double v0 = fma(Z0, P.nvz, nv) * r;
      const float gu = static_cast<float>(P.nuz * r);
      const float gv = static_cast<float>(P.nvz * r);
      if (!(isfinite(u0) && isfinite(v0) && isfinite(gu) && isfinite(gv)))
        continue;
      const float w = rf * rf;
      const double uc0 = fmin(fmax(u0, -1e6), 1e6);
      const double ufl = floor(uc0);
      const int32_t iub = static_cast<int32_t>(ufl);
      const float fu0 = static_cast<float>(uc0 - ufl);
      const double vc0 = fmin(fmax(v0, -1e6), 1e6);
      const double vfl = floor(vc0);
      const int32_t ivb = static_cast<int32_t>(vfl);
      const float fv0 = static_cast<float>(vc0 - vfl);
      uint32_t off[K];
      float fu[K], fv[K];
      const float ku = static_cast<float>(K - 1) * gu;
      const float kv = static_cast<float>(K - 1) * gv;
      const bool inside =
          run_inside(iub, fu0 + fminf(ku, 0.f), fu0 + fmaxf(ku, 0.f), cmax) &&
          run_inside(ivb, fv0 + fminf(kv, 0.f), fv0 + fmaxf(kv, 0.f), rmax);
      if (__all(inside)) {
#pragma unroll
        for (int k = 0; k < K; ++k) {
          const float fk = static_cast<float>(k);
          int32_t iu, iv;
          split_inside(fmaf(fk, gu, fu0), iub, iu, fu[k]);
          split_inside(fmaf(fk, gv, fv0), ivb, iv, fv[k]);
          off[k] = __umul24(static_cast<uint32_t>(iv), trb) +
                   (static_cast<uint32_t>(iu) << 3);
        }
      } else {
        const float ulo = static_cast<float>(-iub);
        const float uup = static_cast<float>(cmax - iub);
        const float vlo = static_cast<float>(-ivb);
        const float vup = static_cast<float>(rmax - ivb);
#pragma unroll
        for (int k = 0; k < K; ++k) {
          const float fk = static_cast<float>(k);
          int32_t iu, iv;
          split_clamped(fmaf(fk, gu, fu0), iub, ulo, uup, iu, fu[k]);
          split_clamped(fmaf(fk, gv, fv0), ivb, vlo, vup, iv, fv[k]);
          off[k] = __umul24(static_cast<uint32_t>(iv), trb) +
                   (static_cast<uint32_t>(iu) << 3);
        }
      }
      kk_float4u tp[K];
#pragma unroll
      for (int k = 0; k < K; ++k) tp[k] = kk_ld4(img, off[k]);
#pragma unroll
      for (int k = 0; k < K; ++k)
        acc[k] = fmaf(w, bilerp(tp[k], fu[k], fv[k]), acc[k]);
    } else if (P.fast) {
      // u and 1/den do not depend on z; v is affine in z
      const float rf = __builtin_amdgcn_rcpf(static_cast<float>(den));
      const double r = refine_rcp(den, rf);
      const double u = nu * r;
      const double v0 = fma(Z0, P.nvz, nv) * r;
      const float gv = static_cast<float>(P.nvz * r);
      // a voxel in the plane of the source parallel to the detector
      // (den = 0) has no projection: skip it
      if (!(isfinite(u) && isfinite(v0) && isfinite(gv))) continue;
      const float w = rf * rf;
      uint32_t iu;
      float fu;
      kk_split_nonneg(fmin(fmax(u, 0.0), static_cast<double>(cmax)), iu, fu);
      const uint32_t offu = iu << 3;
      const double vc0 = fmin(fmax(v0, -1e6), 1e6);
      const double vfl = floor(vc0);
      const int32_t ivb = static_cast<int32_t>(vfl);
      const float fv0 = static_cast<float>(vc0 - vfl);
      const float vlo = static_cast<float>(-ivb);
      const float vup = static_cast<float>(rmax - ivb);
      uint32_t off[K];
      float fv[K];
#pragma unroll
      for (int k = 0; k < K; ++k) {
        int32_t iv;
        split_clamped(fmaf(static_cast<float>(k), gv, fv0), ivb, vlo, vup, iv,
                      fv[k]);
        off[k] = __umul24(static_cast<uint32_t>(iv), trb) + offu;
      }
      kk_float4u tp[K];
#pragma unroll
      for (int k = 0; k < K; ++k) tp[k] = kk_ld4(img, off[k]);
#pragma unroll
      for (int k = 0; k < K; ++k)
        acc[k] = fmaf(w, bilerp(tp[k], fu, fv[k]), acc[k]);
    } else {
      // integer bases at the run's first voxel; per voxel,
      // u(k) - ub = (e0u + k e1u) / den(k) with float32 numerators
      const double den0 = fma(Z0, P.dz, den);
      const double nu0 = fma(Z0, P.nuz, nu);
      const double nv0 = fma(Z0, P.nvz, nv);
      const double r0 = refine_rcp(
          den0, __builtin_amdgcn_rcpf(static_cast<float>(den0)));
      double ub = 0.0, vb = 0.0;
      const double u0 = nu0 * r0, v0 = nv0 * r0;
      if (isfinite(u0) && isfinite(v0)) {
        ub = floor(fmin(fmax(u0, -1e6), 1e6));
        vb = floor(fmin(fmax(v0, -1e6), 1e6));
      }
      const float e0u = static_cast<float>(fma(-ub, den0, nu0));
      const float e1u = static_cast<float>(fma(-ub, P.dz, P.nuz));
      const float e0v = static_cast<float>(fma(-vb, den0, nv0));
      const float e1v = static_cast<float>(fma(-vb, P.dz, P.nvz));
      const float d0f = static_cast<float>(den0);
      const float dzf = static_cast<float>(P.dz);
      const int32_t iub = static_cast<int32_t>(ub);
      const int32_t ivb = static_cast<int32_t>(vb);
      uint32_t off[K];
      float fu[K], fv[K], w[K];
      // the run's end points: with den of one sign along the run, u and v
      // are monotonic in k (ratios of affine forms), so end points inside
      // the detector put the whole run inside (non-finite values fail the
      // comparisons)
      const float kl = static_cast<float>(K - 1);
      const float dK = fmaf(kl, dzf, d0f);
      const float rf0 = __builtin_amdgcn_rcpf(d0f);
      const float rfK = __builtin_amdgcn_rcpf(dK);
      const float du0 = e0u * rf0, duK = fmaf(kl, e1u, e0u) * rfK;
      const float dv0 = e0v * rf0, dvK = fmaf(kl, e1v, e0v) * rfK;
      const bool inside = d0f * dK > 0.f &&
                          run_inside(iub, fminf(du0, duK), fmaxf(du0, duK),
                                     cmax) &&
                          run_inside(ivb, fminf(dv0, dvK), fmaxf(dv0, dvK),
                                     rmax);
      if (__all(inside)) {
#pragma unroll
        for (int k = 0; k < K; ++k) {
          const float fk = static_cast<float>(k);
          const float r = __builtin_amdgcn_rcpf(fmaf(fk, dzf, d0f));
          int32_t iu, iv;
          split_inside(fmaf(fk, e1u, e0u) * r, iub, iu, fu[k]);
          split_inside(fmaf(fk, e1v, e0v) * r, ivb, iv, fv[k]);
          off[k] = __umul24(static_cast<uint32_t>(iv), trb) +
                   (static_cast<uint32_t>(iu) << 3);
          w[k] = r * r;
        }
      } else {
        // a voxel without a finite projection reads index 0 with weight 0
        // (its offset is put at the lower bound)
        const float ulo = static_cast<float>(-iub);
        const float uup = static_cast<float>(cmax - iub);
        const float vlo = static_cast<float>(-ivb);
        const float vup = static_cast<float>(rmax - ivb);
#pragma unroll
        for (int k = 0; k < K; ++k) {
          const float fk = static_cast<float>(k);
          const float r = __builtin_amdgcn_rcpf(fmaf(fk, dzf, d0f));
          const float du = fmaf(fk, e1u, e0u) * r;
          const float dv = fmaf(fk, e1v, e0v) * r;
          const bool ok = isfinite(du) && isfinite(dv);
          int32_t iu, iv;
          split_clamped(ok ? du : ulo, iub, ulo, uup, iu, fu[k]);
          split_clamped(ok ? dv : vlo, ivb, vlo, vup, iv, fv[k]);
          off[k] = __umul24(static_cast<uint32_t>(iv), trb) +
                   (static_cast<uint32_t>(iu) << 3);
          w[k] = ok ? r * r : 0.f;
        }
      }
      kk_float4u tp[K];
#pragma unroll
      for (int k = 0; k < K; ++k) tp[k] = kk_ld4(img, off[k]);
#pragma unroll
      for (int k = 0; k < K; ++k)
        acc[k] = fmaf(w[k], bilerp(tp[k], fu[k], fv[k]), acc[k]);
    }
  }

#pragma unroll
  for (int k = 0; k < K; ++k) {
    if (iz0 + k >= A.nz) break;
    bp_store(A, ix, iy, iz0 + k, acc[k]);
  }
}

// Register caps without spills: 5 wavefronts per SIMD up to 8 voxels per
// thread, 3 at 16 (the unclamped and clamped branches together would
// otherwise take 102 and 176 VGPRs, i.e. 4 and 2 waves).
constexpr int bp_min_blocks(int k) { return k <= 8 ? 5 : 3; }

template <int K>
__global__ __launch_bounds__(256, bp_min_blocks(K)) void cone_bp_kernel(
    const kk::BpAngle* __restrict__ tab, BpArgs A) {
  bp_tile<K, false>(tab, A,
                    kk_xcd_remap(blockIdx.x, A.total_blocks, A.xcd_group));
}


// ---- detector patches in LDS ----------------------------------------------
//
// A workgroup is a tile of 16 x 16 columns of K voxels.  Per angle it stages
// the detector patch that the tile projects onto in LDS (from planes: the
// projections column-major, each column followed by zeros), and every update
// reads its four taps there: two paired reads.  The next angle's patch is on
// its way into registers meanwhile.  Patches of 64 angles are located at a
// time, one angle per lane, from the tile's corners.  Reads outside the
// detector become zeros by the buffer descriptor (columns) and the zeros
// between columns (rows), so nothing is clamped per update.
//
// What bounds circular orbits (MI355X): a gather from global memory costs a CU
// 16 cycles per 64 updates (it took 20 with 16.5 vector instructions beside),
// the two LDS reads 10 and the patch ~3.  Measured: 512^3 / 720 50.8 -> 38.0 ms,
// 256^3 / 360 3.2 -> 2.3 ms, 128^3 / 180 0.25 -> 0.18 ms.  At 512^3 three units
// are near their limits, none at it alone: 190 GB beyond the L2 (patches are
// staged whole, 2.4 times the pair kernel's bytes) at 5.5 TB/s, more than a copy
// reaches; LDS busy in 72% of the cycles, 10% of them bank conflicts; 12.5 vector
// instructions per update, 0.24 per SIMD and cycle (0.25 at four cycles each, which
// plain float32 adds and multiplies undercut).
// * Bank conflicts decide the layout: a wavefront is 8 x 8 columns and the
//   patch pitch 64 + 6 words (512^3: 38.1 ms; pitches 64 + 1, 2, 3, 4, 5, 8,
//   11 and 13: 47.5, 39.1, 37.9, 41.6, 38.1, 59.9, 46.0 and 42.5 ms, and at
//   256^3 64 + 6 is 3% ahead of 64 + 3; a wavefront of 16 x 4 columns: 41).
// * K = 16: runs of 8 and 24 took 71 and 38.9 ms (at 256^3 4.0 and 2.8).
// * SPLIT > 1: the angles are dealt to that many groups of 256 threads and
//   the groups' sums added at the end, where the tiles alone leave the chip
//   idle (128^3: 0.244, 0.179 and 0.194 ms with 1, 2 and 4 parts).
//
// CIRC, circular orbits: the column and the weight are the same for a run of
// K voxels, and the row of an update is 64-bit fixed point (32 fraction bits),
// stepped by one 64-bit add per voxel.
//
// Otherwise (plans with a general angle): column, row and weight per voxel,
// from float32 numerators around an integer base in the middle of the run and
// one reciprocal.  24 vector instructions per update bound it (0.28 per SIMD and
// cycle; LDS busy in 42% of the cycles; the pair kernel's gather took as long as its
// instructions): 256^3 / 360 wobbling angles 4.9 -> 3.8 ms, 128^3 / 128
// 0.27 -> 0.20 ms.  Five wavefronts per SIMD instead of four spill: 3.84 ms.
// The reciprocal as a series around the base and addresses made in float32 were
// no faster (3.9 ms).
constexpr int kPatchRun = 16;                  // K
constexpr int kPatchLanes = 64;                // rows per patch column
constexpr int kPatchPitch = kPatchLanes + 6;   // LDS words per column
constexpr int kPatchCols = 64;
constexpr int kPatchGap = KK_PLANE_GAP;        // zero rows after a column
static_assert(kPatchGap >= kPatchLanes, "a patch column ends in its own gap");

// x as 64-bit fixed point with 32 fraction bits, |x| < 2^19: the mantissa of
// x + 1.5 * 2^20.  The high word carries kFixedHi besides.
constexpr double kFixedMagic = 1572864.0;
constexpr uint32_t kFixedHi = 0x41380000u;
__device__ __forceinline__ uint64_t fixed_bits(double x) {
  return __builtin_bit_cast(uint64_t, x + kFixedMagic);
}

template <int K, int SPLIT, bool CIRC>
__global__ __launch_bounds__(256 * SPLIT, CIRC ? 5 : 4) void
cone_bp_patch_kernel(
    const kk::BpAngle* __restrict__ tab, BpArgs A) {
  typedef __attribute__((address_space(3))) const float* lds_ptr;
  __shared__ float patch_s[SPLIT][kPatchCols * kPatchPitch];
  int32_t tx, ty, tz;
  if (!bp_decode(A, kk_xcd_remap(blockIdx.x, A.total_blocks, A.xcd_group), tx,
                 ty, tz))
    return;  // the whole workgroup
  const int32_t lane = int32_t(threadIdx.x) & 63;
  const int32_t sub = __builtin_amdgcn_readfirstlane(int32_t(threadIdx.x) >> 8);
  const int32_t wave =
      __builtin_amdgcn_readfirstlane((int32_t(threadIdx.x) >> 6) & 3);
  const int32_t tid = int32_t(threadIdx.x) & 255;
  // a wavefront is 8 x 8 columns
  const int32_t ix = tx * 16 + (tid & 7) + ((tid >> 3) & 8);
  const int32_t iy = ty * 16 + ((tid >> 3) & 7) + ((tid >> 4) & 8);
  const int32_t iz0 = tz * K;
  // columns outside the volume repeat its last ones (not written)
  const double X = min(ix, A.nx - 1) - 0.5 * A.nx + 0.5;
  const double Y = min(iy, A.ny - 1) - 0.5 * A.ny + 0.5;
  const double Z0 = iz0 - 0.5 * A.nz + 0.5;
  float* patch = patch_s[sub];
  const uint32_t patch_at = __builtin_amdgcn_readfirstlane(
      static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_ptr)patch)));
  const int32_t pitch = static_cast<int32_t>(A.trb);  // bytes per column

  float acc[K];
#pragma unroll
  for (int k = 0; k < K; ++k) acc[k] = 0.f;
  // patches of 64 of this part's angles at a time, one per lane: origin
  // column and row, number of columns (0: the tile projects off the detector)
  int32_t pc = 0, pr = 0, pn = 0;
  auto bounds = [&](int32_t a) {
    pn = 0;
    if (a >= A.n_angles) return;
    const kk::BpAngle& P = tab[a];
    // (from integers, here: kept in registers they would cost the loop)
    int32_t ex = tx * 16, ey = ty * 16;
    asm volatile("" : "+v"(ex), "+v"(ey));
    double ul = 1e30, uh = -1e30, vl = 1e30, vh = -1e30;
#pragma unroll 1
    for (int e = 0; e < (CIRC ? 4 : 8); ++e) {
      const double x =
          min(ex + (e & 1 ? 15 : 0), A.nx - 1) - 0.5 * A.nx + 0.5;
      const double y =
          min(ey + (e & 2 ? 15 : 0), A.ny - 1) - 0.5 * A.ny + 0.5;
      double d = fma(y, P.dy, fma(x, P.dx, P.dw));
      double nu = fma(y, P.nuy, fma(x, P.nux, P.nuw));
      const double z = CIRC || e < 4 ? Z0 : Z0 + (K - 1);
      if constexpr (!CIRC) {
        d = fma(z, P.dz, d);
        nu = fma(z, P.nuz, nu);
      }
      const double r =
          refine_rcp(d, __builtin_amdgcn_rcpf(static_cast<float>(d)));
      const double u = nu * r;
      const double v = fma(z, P.nvz, fma(y, P.nvy, fma(x, P.nvx, P.nvw))) * r;
      const double w =
          CIRC ? fma(static_cast<double>(K - 1), P.nvz * r, v) : v;
      ul = fmin(ul, u);
      uh = fmax(uh, u);
      vl = fmin(vl, fmin(v, w));
      vh = fmax(vh, fmax(v, w));
    }
    // (without the halo that the padded coordinates count; the widening
    // covers the rounding of the threads' own coordinates: float64, or
    // float32 offsets of up to 64 texels)
    constexpr double kWide = CIRC ? 1e-6 : 1e-4;
    const double c0 = floor(ul - kWide) - kk::kHaloLo;
    const double r0 = floor(vl - kWide) - kk::kHaloLo;
    const double c1 = floor(uh + kWide) - kk::kHaloLo + 1;
    const double r1 = floor(vh + kWide) - kk::kHaloLo + 1;
    if (c1 < 0 || c0 >= A.cols || r1 < 0 || r0 >= A.rows) return;
    pc = static_cast<int32_t>(c0);
    pr = static_cast<int32_t>(r0);
    pn = static_cast<int32_t>(c1 - c0) + 1;
  };
  // (the compiler would otherwise wait for all loads wherever the registers
  // of these are used again)
  auto settle = [] { __builtin_amdgcn_s_waitcnt(0x0f70); };  // vmcnt(0)
  constexpr int NS = kPatchCols / 4;
  float st[NS];
  int32_t c0 = 0, r0 = 0, nc = 0;   // the staged patch
  auto stage = [&](int32_t a, int32_t l) {
    c0 = __builtin_amdgcn_readlane(pc, l);
    r0 = __builtin_amdgcn_readlane(pr, l);
    nc = __builtin_amdgcn_readlane(pn, l);
    if (nc == 0) return;
    const auto rsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<char*>(A.tex) + static_cast<uint64_t>(a) * A.tab_b, 0,
        static_cast<int32_t>(A.tab_b), 0x00020000);
    uint32_t o = static_cast<uint32_t>((c0 + wave) * pitch + (r0 + lane) * 4);
#pragma unroll
    for (int j = 0; j < NS; ++j) {
      if (wave + 4 * j >= nc) break;
      asm volatile("" : "+v"(o));
      st[j] = __builtin_bit_cast(
          float, __builtin_amdgcn_raw_buffer_load_b32(rsrc, o, 0, 0));
      o += 4 * pitch;
    }
  };
  const int32_t mine = (A.n_angles - sub + SPLIT - 1) / SPLIT;
  const int32_t most = (A.n_angles + SPLIT - 1) / SPLIT;
  bounds(sub + lane * SPLIT);
  settle();
  stage(sub, 0);
  for (int32_t q = 0; q < most; ++q) {
    const int32_t a = sub + q * SPLIT;
    const int32_t cc = c0, cr = r0, n = q < mine ? nc : 0;
    __syncthreads();  // the previous patch has been read
#pragma unroll
    for (int j = 0; j < NS; ++j) {
      if (wave + 4 * j >= n) break;
      patch[(wave + 4 * j) * kPatchPitch + lane] = st[j];
    }
    __syncthreads();
    if (q + 1 < mine) {
      if (((q + 1) & 63) == 0) {
        bounds(a + SPLIT + lane * SPLIT);
        settle();
      }
      stage(a + SPLIT, (q + 1) & 63);
    }
    if (n == 0) continue;
    const kk::BpAngle& P = tab[a];
    const double den = fma(Y, P.dy, fma(X, P.dx, P.dw));
    const double nu = fma(Y, P.nuy, fma(X, P.nux, P.nuw));
    const double nv = fma(Y, P.nvy, fma(X, P.nvx, P.nvw));
    if constexpr (CIRC) {
      const float rf = __builtin_amdgcn_rcpf(static_cast<float>(den));
      const double r = refine_rcp(den, rf);
      const double u = fma(nu, r, -static_cast<double>(cc + kk::kHaloLo));
      uint32_t iu;
      float fu;
      kk_split_nonneg(u, iu, fu);
      const double v0 =
          fma(fma(Z0, P.nvz, nv), r, -static_cast<double>(cr + kk::kHaloLo));
      uint64_t V = fixed_bits(v0);
      const uint64_t G = fixed_bits(P.nvz * r) -
                         (static_cast<uint64_t>(kFixedHi) << 32);
      const float w = rf * rf;
      const uint32_t at =
          patch_at + __umul24(iu, kPatchPitch * 4u) - (kFixedHi << 2);
#pragma unroll
      for (int k = 0; k < K; ++k) {
        uint32_t p;  // one shift-add of the row (not a 64-bit shift)
        asm("v_lshl_add_u32 %0, %1, 2, %2"
            : "=v"(p)
            : "v"(static_cast<uint32_t>(V >> 32)), "v"(at));
        const lds_ptr t = (lds_ptr)p;
        const float l0 = fmaf(fu, t[kPatchPitch] - t[0], t[0]);
        const float l1 = fmaf(fu, t[kPatchPitch + 1] - t[1], t[1]);
        const float fv =
            static_cast<float>(static_cast<uint32_t>(V)) * 0x1p-32f;
        acc[k] = fmaf(w, fmaf(fv, l1 - l0, l0), acc[k]);
        V += G;
        // (four voxels' reads in flight, within the register cap)
        if (k % 4 == 3) __builtin_amdgcn_sched_barrier(0);
      }
    } else {
      // Integer bases at the middle of the run (its ends are then as close
      // as those of a run half as long), relative to the patch; per voxel,
      // u(k) - ub = (e0u + (k - K / 2) e1u) / den(k), float32 numerators.
      const double Zm = Z0 + K / 2;
      const double den0 = fma(Zm, P.dz, den);
      const double nu0 = fma(Zm, P.nuz, nu);
      const double nv0 = fma(Zm, P.nvz, nv);
      const double r0 = refine_rcp(
          den0, __builtin_amdgcn_rcpf(static_cast<float>(den0)));
      const double ub = floor(nu0 * r0), vb = floor(nv0 * r0);
      const float e0u = static_cast<float>(fma(-ub, den0, nu0));
      const float e1u = static_cast<float>(fma(-ub, P.dz, P.nuz));
      const float e0v = static_cast<float>(fma(-vb, den0, nv0));
      const float e1v = static_cast<float>(fma(-vb, P.dz, P.nvz));
      const float d0f = static_cast<float>(den0);
      const float dzf = static_cast<float>(P.dz);
      const int32_t at =
          static_cast<int32_t>(patch_at) +
          (static_cast<int32_t>(ub) - cc - kk::kHaloLo) * (kPatchPitch * 4) +
          (static_cast<int32_t>(vb) - cr - kk::kHaloLo) * 4;
#pragma unroll
      for (int k = 0; k < K; ++k) {
        const float fk = static_cast<float>(k - K / 2);
        const float r = __builtin_amdgcn_rcpf(fmaf(fk, dzf, d0f));
        const float du = fmaf(fk, e1u, e0u) * r;
        const float dv = fmaf(fk, e1v, e0v) * r;
        const float lu = floorf(du), lv = floorf(dv);
        const float fu = du - lu, fv = dv - lv;
        // (small integers: exact)
        const int32_t i = static_cast<int32_t>(
            fmaf(lu, static_cast<float>(kPatchPitch), lv));
        uint32_t p;
        asm("v_lshl_add_u32 %0, %1, 2, %2" : "=v"(p) : "v"(i), "v"(at));
        const lds_ptr t = (lds_ptr)p;
        const float l0 = fmaf(fu, t[kPatchPitch] - t[0], t[0]);
        const float l1 = fmaf(fu, t[kPatchPitch + 1] - t[1], t[1]);
        acc[k] = fmaf(r * r, fmaf(fv, l1 - l0, l0), acc[k]);
        if (k % 4 == 3) __builtin_amdgcn_sched_barrier(0);
      }
    }
  }

  if constexpr (SPLIT == 1) {
    if (ix >= A.nx || iy >= A.ny) return;
#pragma unroll
    for (int k = 0; k < K; ++k) {
      if (iz0 + k >= A.nz) break;
      bp_store(A, ix, iy, iz0 + k, acc[k]);
    }
  } else {
    // the parts' sums, in order; every part writes K / SPLIT of the run
    static_assert(K % SPLIT == 0 && 256 * K <= kPatchCols * kPatchPitch,
                  "a part's sums take its patch");
    __syncthreads();
#pragma unroll
    for (int k = 0; k < K; ++k) patch[k * 256 + tid] = acc[k];
    __syncthreads();
    if (ix >= A.nx || iy >= A.ny) return;
#pragma unroll
    for (int k = 0; k < K / SPLIT; ++k) {
      const int32_t z = sub * (K / SPLIT) + k;
      if (iz0 + z >= A.nz) break;
      float sum = patch_s[0][z * 256 + tid];
#pragma unroll
      for (int p = 1; p < SPLIT; ++p) sum += patch_s[p][z * 256 + tid];
      bp_store(A, ix, iy, iz0 + z, sum);
    }
  }
}

struct BpItem {
  const kk::BpAngle* tab;
  BpArgs args;
};

// Many problems, one persistent launch (see cone_fp_batch_kernel).
template <int K>
__global__ __launch_bounds__(256, bp_min_blocks(K)) void cone_bp_batch_kernel(
    const BpItem* __restrict__ items, const int64_t* __restrict__ first,
    int32_t n, int64_t total) {
  for (int64_t g = blockIdx.x; g < total; g += gridDim.x) {
    int32_t lo = 0, hi = n - 1;
    while (lo < hi) {
      const int32_t mid = (lo + hi + 1) >> 1;
      if (first[mid] <= g)
        lo = mid;
      else
        hi = mid - 1;
    }
    const BpItem& it = items[lo];
    const int64_t local = g - first[lo];
    bp_tile<K, true>(it.tab, it.args,
               kk_xcd_remap(local, it.args.total_blocks, it.args.xcd_group));
  }
}

}  // namespace

namespace {

// Validate one backprojection problem and fill its kernel arguments for
// z-runs of `zrun` voxels.
int make_bp_args(const kk::BpSpec& S, int32_t zrun, BpArgs& A) {
  using namespace kk;
  if (S.plan == nullptr || !S.plan->bp_set)
    return fail(KK_ERR_NOT_SET,
                "Please set the parameters with `set_params()`.");
  if (S.tex == nullptr || S.out == nullptr)
    return fail(KK_ERR_INVALID, "kk_cone_bp: null argument");
  if (S.n_angles != S.plan->bp_n)
    return fail(KK_ERR_SHAPE,
                "kk_cone_bp: %d projections but parameters for %d angles",
                S.n_angles, S.plan->bp_n);
  if (S.rows <= 0 || S.cols <= 0 || S.shape[0] <= 0 || S.shape[1] <= 0 ||
      S.shape[2] <= 0)
    return fail(KK_ERR_INVALID, "kk_cone_bp: bad sizes");
  if (zrun != 4 && zrun != 8 && zrun != 16)
    return fail(KK_ERR_INVALID, "kk_cone_bp: z-run must be 4, 8 or 16");
  const int64_t trb = int64_t(S.cols + kHalo) * 8;
  const int64_t tab_b = int64_t(S.rows + kHalo) * trb;
  if (tab_b >= (int64_t(1) << 32) || trb >= (int64_t(1) << 24))
    return fail(KK_ERR_UNSUPPORTED, "kk_cone_bp: detector too large");
  if (S.mode == 2 && S.C == nullptr)
    return fail(KK_ERR_INVALID, "kk_cone_bp: SIRT update needs C");
  A = BpArgs{};
  A.tex = reinterpret_cast<const char*>(S.tex);
  A.tab_b = uint32_t(tab_b);
  A.trb = uint32_t(trb);
  A.nx = S.shape[0];
  A.ny = S.shape[1];
  A.nz = S.shape[2];
  A.n_angles = S.plan->bp_n;
  A.rows = S.rows;
  A.cols = S.cols;
  A.out = S.out;
  A.vs0 = S.vs[0];
  A.vs1 = S.vs[1];
  A.vs2 = S.vs[2];
  A.scale = S.scale;
  A.mode = S.mode;
  if (S.mode == 2) {
    A.C = S.C;
    A.cs0 = S.cs[0];
    A.cs1 = S.cs[1];
    A.cs2 = S.cs[2];
    A.mask = S.mask;
    if (S.mask) {
      A.ms0 = S.ms[0];
      A.ms1 = S.ms[1];
      A.ms2 = S.ms[2];
    }
    A.lo = S.lo;
    A.hi = S.hi;
    A.clip_lo = S.clip_lo;
    A.clip_hi = S.clip_hi;
    A.xtex = S.xtex;
    if (S.xtex) {
      // voxel (x, y, z) in frame a: element (c_a, c_b + 1, c_c + 1)
      // component 0 and element (c_a, c_b, c_c + 1) component 1
      int64_t off = 0;  // floats
      for (int a = 0; a < 3; ++a) {
        if (!(S.xtex_mask & (1 << a))) continue;
        const int b = kFrameB[a], c = kFrameC[a];
        const int64_t tcn = S.shape[c] + kHalo, tbn = S.shape[b] + kHalo;
        int64_t ws[3];
        ws[a] = 2 * tbn * tcn;
        ws[b] = 2 * tcn;
        ws[c] = 2;
        const int f = A.n_frames++;
        A.fr_origin[f] = off + 2 * (kHaloLo * tcn + kHaloLo);
        A.fr_s0[f] = ws[0];
        A.fr_s1[f] = ws[1];
        A.fr_s2[f] = ws[2];
        A.fr_dual[f] = 1 - 2 * tcn;
        off += 2 * frame_elems(S.shape, a);
      }
    }
  }
  A.tiles_x = (A.nx + 15) / 16;
  A.tiles_y = (A.ny + 15) / 16;
  A.tiles_z = (A.nz + zrun - 1) / zrun;
  // Circular orbits, tile counts divisible by 4: groups of 4 x 4 x 4
  // tiles, each group's ids on one XCD; neighbouring tiles project onto
  // overlapping detector patches, which that XCD's L2 then serves
  // (measured at 512^3 / 720 angles: 51.5 ms, against 53.3 ms for runs of
  // 16 tiles along x; 4 x 4 x 8, 8 x 4 x 4, 4 x 4 x 2 and 4 x 4 x 16 took
  // 52.2, 51.7, 52.1 and 52.6 ms).  Other geometries keep runs of 16
  // tiles along x per XCD (1.5% faster than round-robin at 512^3): the
  // groups made the tilted-detector batches of the batching workload
  // slower (its batched backprojection 57.1 -> 65.8 ms).
  const bool groups = S.plan->bp_all_circ && A.tiles_x % 4 == 0 &&
                      A.tiles_y % 4 == 0 && A.tiles_z % 4 == 0;
  A.gx = A.gy = A.gz = groups ? 4 : 1;
  A.xcd_group = groups ? 64 : 16;
  A.total_blocks = int64_t(A.tiles_x) * A.tiles_y * A.tiles_z;
  if (A.total_blocks >= (int64_t(1) << 31))
    return fail(KK_ERR_UNSUPPORTED, "kk_cone_bp: grid too large");
  return KK_OK;
}

int launch_bp_spec(const kk::BpSpec& S, int32_t zrun, hipStream_t stream) {
  BpArgs A;
  const int rc = make_bp_args(S, zrun, A);
  if (rc != KK_OK) return rc;
  const dim3 grid(unsigned(A.total_blocks)), block(256);
  switch (zrun) {
    case 4:
      hipLaunchKernelGGL(cone_bp_kernel<4>, grid, block, 0, stream,
                         S.plan->bp, A);
      break;
    case 8:
      hipLaunchKernelGGL(cone_bp_kernel<8>, grid, block, 0, stream,
                         S.plan->bp, A);
      break;
    default:
      hipLaunchKernelGGL(cone_bp_kernel<16>, grid, block, 0, stream,
                         S.plan->bp, A);
      break;
  }
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return kk::hip_fail(e, "cone_bp_kernel");
  return KK_OK;
}

}  // namespace

namespace kk {

struct BpBatch {
  BpItem* items = nullptr;
  int64_t* first = nullptr;
  int32_t n = 0;
  int64_t total = 0;
  int32_t zrun = 8;
};

int bp_batch_build(const std::vector<BpSpec>& specs, int32_t zrun,
                   BpBatch** out) {
  if (specs.empty()) return fail(KK_ERR_INVALID, "empty backprojection batch");
  if (zrun != 4 && zrun != 8 && zrun != 16) zrun = 8;
  std::vector<BpItem> items(specs.size());
  std::vector<int64_t> first(specs.size());
  int64_t total = 0;
  for (size_t p = 0; p < specs.size(); ++p) {
    const int rc = make_bp_args(specs[p], zrun, items[p].args);
    if (rc != KK_OK) return rc;
    items[p].tab = specs[p].plan->bp;
    first[p] = total;
    total += items[p].args.total_blocks;
  }
  auto* b = new (std::nothrow) BpBatch();
  if (b == nullptr) return fail(KK_ERR_INVALID, "out of host memory");
  b->n = static_cast<int32_t>(specs.size());
  b->total = total;
  b->zrun = zrun;
  hipError_t e = hipMalloc(&b->items, sizeof(BpItem) * items.size());
  if (e == hipSuccess) e = hipMalloc(&b->first, sizeof(int64_t) * first.size());
  if (e == hipSuccess)
    e = hipMemcpy(b->items, items.data(), sizeof(BpItem) * items.size(),
                  hipMemcpyHostToDevice);
  if (e == hipSuccess)
    e = hipMemcpy(b->first, first.data(), sizeof(int64_t) * first.size(),
                  hipMemcpyHostToDevice);
  if (e != hipSuccess) {
    bp_batch_free(b);
    return hip_fail(e, "backprojection batch descriptors");
  }
  *out = b;
  return KK_OK;
}

void bp_batch_free(BpBatch* b) {
  if (b == nullptr) return;
  if (b->items) hipFree(b->items);
  if (b->first) hipFree(b->first);
  delete b;
}

int bp_batch_launch(const BpBatch* b, int32_t grid_blocks,
                    hipStream_t stream) {
  if (b == nullptr) return fail(KK_ERR_NOT_SET, "backprojection batch not built");
  int64_t g = grid_blocks > 0 ? grid_blocks : b->total;
  if (g > b->total) g = b->total;
  if (g <= 0) return KK_OK;
  const dim3 grid(static_cast<unsigned>(g)), block(256);
  switch (b->zrun) {
    case 4:
      hipLaunchKernelGGL(cone_bp_batch_kernel<4>, grid, block, 0, stream,
                         b->items, b->first, b->n, b->total);
      break;
    case 8:
      hipLaunchKernelGGL(cone_bp_batch_kernel<8>, grid, block, 0, stream,
                         b->items, b->first, b->n, b->total);
      break;
    default:
      hipLaunchKernelGGL(cone_bp_batch_kernel<16>, grid, block, 0, stream,
                         b->items, b->first, b->n, b->total);
      break;
  }
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return hip_fail(e, "cone_bp_batch_kernel");
  return KK_OK;
}

}  // namespace kk

namespace {

int fill_bp_spec(kk::BpSpec& S, const kk_plan* plan, const float* tex,
                 int32_t n_angles, int32_t rows, int32_t cols, float* vol,
                 const int32_t shape[3], const int64_t vs[3], float scale,
                 int32_t mode) {
  if (shape == nullptr || vs == nullptr)
    return kk::fail(KK_ERR_INVALID, "kk_cone_bp: null argument");
  S.plan = plan;
  S.tex = tex;
  S.n_angles = n_angles;
  S.rows = rows;
  S.cols = cols;
  S.out = vol;
  for (int t = 0; t < 3; ++t) {
    S.shape[t] = shape[t];
    S.vs[t] = vs[t];
  }
  S.scale = scale;
  S.mode = mode;
  return KK_OK;
}

int fill_sirt_update(kk::BpSpec& S, const float* C, const int64_t cs[3],
                     const float* mask, const int64_t ms[3], float lo,
                     float hi, int32_t clip_lo, int32_t clip_hi, float* x_tex,
                     int32_t x_tex_mask) {
  if (C == nullptr || cs == nullptr)
    return kk::fail(KK_ERR_INVALID, "kk_sirt_bp_update: C is required");
  if (mask != nullptr && ms == nullptr)
    return kk::fail(KK_ERR_INVALID, "kk_sirt_bp_update: mask strides");
  if (x_tex != nullptr && (x_tex_mask <= 0 || x_tex_mask > 7))
    return kk::fail(KK_ERR_INVALID, "kk_sirt_bp_update: texture mask");
  S.C = C;
  S.mask = mask;
  for (int t = 0; t < 3; ++t) {
    S.cs[t] = cs[t];
    S.ms[t] = mask ? ms[t] : 0;
  }
  S.lo = lo;
  S.hi = hi;
  S.clip_lo = clip_lo;
  S.clip_hi = clip_hi;
  S.xtex = x_tex;
  S.xtex_mask = x_tex ? x_tex_mask : 0;
  return KK_OK;
}

}  // namespace

namespace kk {

int bp_spec(BpSpec& S, const kk_plan* plan, const float* tex,
            int32_t n_angles, int32_t rows, int32_t cols, float* vol,
            const int32_t shape[3], const int64_t vs[3], float scale,
            int32_t additive) {
  return fill_bp_spec(S, plan, tex, n_angles, rows, cols, vol, shape, vs,
                      scale, additive ? 1 : 0);
}

int sirt_update_spec(BpSpec& S, const kk_plan* plan, const float* res_tex,
                     int32_t n_angles, int32_t rows, int32_t cols, float* x,
                     const int32_t shape[3], const int64_t xs[3],
                     const float* C, const int64_t cs[3], const float* mask,
                     const int64_t ms[3], float lo, float hi,
                     int32_t clip_lo, int32_t clip_hi, float* x_tex,
                     int32_t x_tex_mask, float scale) {
  int rc = fill_bp_spec(S, plan, res_tex, n_angles, rows, cols, x, shape, xs,
                        scale, 2);
  if (rc != KK_OK) return rc;
  return fill_sirt_update(S, C, cs, mask, ms, lo, hi, clip_lo, clip_hi,
                          x_tex, x_tex_mask);
}

}  // namespace kk

namespace {

// Largest |du/dx| + |du/dy| (and v alike) over the volume's columns for a
// coordinate f = num / den of affine forms in (x, y): df/dx = ((nx dy - ny dx)
// y + nx dw - nw dx) / den^2 is monotonic in x and has at most one extremum in
// y between the ends (df/dy alike).
double steepest(double nx, double ny, double nw, double dx, double dy,
                double dw, double hx, double hy) {
  auto partial = [&](double n1, double n2, double d1, double d2, double h1,
                     double h2) {  // d/dx1, (x1, x2) in [-h1, h1] x [-h2, h2]
    const double A = n1 * d2 - n2 * d1, B = n1 * dw - nw * d1;
    double most = 0.0;
    for (int e = 0; e < 2; ++e) {
      const double c = dw + d1 * (e ? h1 : -h1);
      const double at[3] = {-h2, h2,
                            A * d2 != 0.0 ? (A * c - 2.0 * d2 * B) / (d2 * A)
                                          : 0.0};
      for (double x2 : at) {
        if (!(std::fabs(x2) <= h2)) continue;
        const double den = c + d2 * x2;
        most = std::fmax(most, std::fabs((A * x2 + B) / (den * den)));
      }
    }
    return most;
  };
  return partial(nx, ny, dx, dy, hx, hy) + partial(ny, nx, dy, dx, hy, hx);
}

// Bounds of the columns and rows of the patch of any tile at any angle
// (ext[0], ext[1]; the host table in `tab`); false where a denominator may
// vanish over the volume or coordinates leave the kernel's ranges, and for
// plans without a general angle that are not circular orbits (detectors
// tilted in their own plane keep the pair kernel, whose arithmetic the
// batched launches share).
bool patch_extent(const std::vector<kk::BpAngle>& tab, const int32_t shape[3],
                  double ext[2]) {
  ext[0] = ext[1] = 0.0;
  if (tab.empty()) return false;
  for (int t = 0; t < 3; ++t)
    if (shape[t] <= 0 || shape[t] > 65536) return false;
  bool circ = true, general = false;
  for (const kk::BpAngle& e : tab) {
    circ = circ && e.fast == 1;
    general = general || e.fast == 0;
  }
  if (!circ && !general) return false;
  const double hx = 0.5 * (shape[0] - 1), hy = 0.5 * (shape[1] - 1);
  const double hz = 0.5 * shape[2] + kPatchRun;
  for (const kk::BpAngle& e : tab) {
    double least = INFINITY, most = 0.0;
    double ul = INFINITY, uh = -INFINITY, vl = INFINITY, vh = -INFINITY;
    bool pos = true, neg = true;
    for (int k = 0; k < 8; ++k) {
      const double x = k & 1 ? hx : -hx, y = k & 2 ? hy : -hy;
      const double z = k & 4 ? hz : -hz;
      const double d = e.dw + e.dx * x + e.dy * y + e.dz * z;
      pos = pos && d > 0.0;
      neg = neg && d < 0.0;
      least = std::fmin(least, std::fabs(d));
      most = std::fmax(most, std::fabs(d));
      const double u = (e.nuw + e.nux * x + e.nuy * y + e.nuz * z) / d;
      const double v = (e.nvw + e.nvx * x + e.nvy * y + e.nvz * z) / d;
      if (!(std::fabs(u) < 1e5) || !(std::fabs(v) < 1e5)) return false;
      ul = std::fmin(ul, u);
      uh = std::fmax(uh, u);
      vl = std::fmin(vl, v);
      vh = std::fmax(vh, v);
    }
    if (!(pos || neg) || !(least > 1e-6 * most)) return false;
    // 15 voxels along each axis; three texels for the ends' floors and the
    // second tap, and rounding
    if (circ) {
      const double du =
          steepest(e.nux, e.nuy, e.nuw, e.dx, e.dy, e.dw, hx, hy);
      double dv = 0.0;
      for (int k = 0; k < 2; ++k)
        dv = std::fmax(dv, steepest(e.nvx, e.nvy,
                                    e.nvw + (k ? hz : -hz) * e.nvz, e.dx,
                                    e.dy, e.dw, hx, hy));
      const double run = (kPatchRun - 1) * std::fabs(e.nvz) / least;
      ext[0] = std::fmax(ext[0], 15.0 * du + 3.01);
      ext[1] = std::fmax(ext[1], 15.0 * dv + run + 3.01);
    } else {
      // between points p and q of f = N / D (affine forms, D of one sign, so
      // f lies between its least and greatest value at the volume's
      // corners): f(q) - f(p) = (N' - f(p) D')(q - p) / D(q)
      auto most_of = [&](double n, double d, double lo, double hi) {
        return std::fmax(std::fabs(n - lo * d), std::fabs(n - hi * d));
      };
      const double du = most_of(e.nux, e.dx, ul, uh) +
                        most_of(e.nuy, e.dy, ul, uh) +
                        most_of(e.nuz, e.dz, ul, uh);
      const double dv = most_of(e.nvx, e.dx, vl, vh) +
                        most_of(e.nvy, e.dy, vl, vh) +
                        most_of(e.nvz, e.dz, vl, vh);
      ext[0] = std::fmax(ext[0], 15.0 * du / least + 3.01);
      ext[1] = std::fmax(ext[1], 15.0 * dv / least + 3.01);
    }
  }
  return true;
}

// Whether the patch kernel is the faster one for the volume's tiles: not where
// half of its only layer of tiles is empty and there are more tiles than CUs to
// hide that (180 angles, patch and pair kernel in us, x = y and z: circular
// (512, 8) 310 and 205, (384, 8) 281 and 186, (512, 9) 310 and 376, (256, 8) 101
// and 176; general (512, 8) 477 and 387, (384, 8) 381 and 317, (512, 9) 478 and
// 681).
bool patches_pay(const int32_t shape[3]) {
  const int64_t cols = ((int64_t(shape[0]) + 15) / 16) *
                       ((int64_t(shape[1]) + 15) / 16);
  return shape[2] > kPatchRun / 2 || cols <= 256;
}

// Whether every patch fits kPatchCols columns and kPatchLanes rows, and the
// patches pay.  The answer for the last detector and volume is kept with the
// plan.
bool patches_fit(const kk_plan_s& plan, int32_t rows, int32_t cols,
                 const int32_t shape[3]) {
  if (rows <= 0 || cols <= 0) return false;
  if (int64_t(rows + kPatchGap) * cols * 4 >= (int64_t(1) << 31)) return false;
  const std::lock_guard<std::mutex> hold(plan.bp_patch_lock);
  if (plan.bp_patch_fits < 0 ||
      !std::equal(shape, shape + 3, plan.bp_patch_shape)) {
    double ext[2];
    const bool ok = patch_extent(plan.bp_host, shape, ext);
    plan.bp_patch_fits =
        ok && ext[0] <= kPatchCols && ext[1] <= kPatchLanes &&
                patches_pay(shape)
            ? 1
            : 0;
    std::copy(shape, shape + 3, plan.bp_patch_shape);
  }
  return plan.bp_patch_fits == 1;
}

int launch_bp_planes(const kk::BpSpec& S, hipStream_t stream) {
  BpArgs A;
  const int rc = make_bp_args(S, kPatchRun, A);
  if (rc != KK_OK) return rc;
  if (!patches_fit(*S.plan, S.rows, S.cols, S.shape))
    return kk::fail(KK_ERR_UNSUPPORTED,
                    "kk_cone_bp_planes: not a geometry for planes (see "
                    "kk_bp_reads_planes)");
  const int64_t pitch = int64_t(S.rows + kPatchGap) * 4;
  A.trb = uint32_t(pitch);
  A.tab_b = uint32_t(pitch * S.cols);
  // parts so that a CU (of 256) holds at least four wavefronts per SIMD
  const int64_t per_cu = (A.total_blocks + 255) / 256;
  const dim3 grid(unsigned(A.total_blocks));
  const int32_t parts = per_cu >= 4 ? 1 : per_cu >= 2 ? 2 : 4;
  auto launch = [&](auto circ) {
    constexpr bool C = decltype(circ)::value;
    auto* kernel = parts == 1   ? &cone_bp_patch_kernel<kPatchRun, 1, C>
                   : parts == 2 ? &cone_bp_patch_kernel<kPatchRun, 2, C>
                                : &cone_bp_patch_kernel<kPatchRun, 4, C>;
    hipLaunchKernelGGL(kernel, grid, dim3(256 * parts), 0, stream, S.plan->bp,
                       A);
  };
  if (S.plan->bp_all_circ)
    launch(std::true_type{});
  else
    launch(std::false_type{});
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return kk::hip_fail(e, "cone_bp_patch_kernel");
  return KK_OK;
}

}  // namespace

extern "C" int32_t kk_bp_reads_planes(const kk_plan* plan, int32_t rows,
                                      int32_t cols, const int32_t shape[3]) {
  if (plan == nullptr || !plan->bp_set || shape == nullptr) return 0;
  return patches_fit(*plan, rows, cols, shape) ? 1 : 0;
}

extern "C" int kk_bp_patch_extent(const double* params, int32_t n,
                                  const int32_t shape[3], double out[2]) {
  if (shape == nullptr || out == nullptr)
    return kk::fail(KK_ERR_INVALID, "kk_bp_patch_extent: null");
  std::vector<kk::BpAngle> tab;
  const int rc = kk::bp_table_host(params, n, tab);
  if (rc != KK_OK) return rc;
  if (!patch_extent(tab, shape, out)) out[0] = out[1] = -1.0;
  return KK_OK;
}

extern "C" int kk_cone_bp_planes(const kk_plan* plan, const float* planes,
                                 int32_t n_angles, int32_t rows, int32_t cols,
                                 float* vol, const int32_t shape[3],
                                 const int64_t vs[3], float output_scale,
                                 int32_t additive, void* stream) {
  kk::BpSpec S;
  const int rc = kk::bp_spec(S, plan, planes, n_angles, rows, cols, vol,
                             shape, vs, output_scale, additive);
  if (rc != KK_OK) return rc;
  return launch_bp_planes(S, static_cast<hipStream_t>(stream));
}

extern "C" int kk_sirt_bp_update_planes(
    const kk_plan* plan, const float* planes, int32_t n_angles, int32_t rows,
    int32_t cols, float* x, const int32_t shape[3], const int64_t xs[3],
    const float* C, const int64_t cs[3], const float* mask,
    const int64_t ms[3], float lo, float hi, int32_t clip_lo, int32_t clip_hi,
    float output_scale, void* stream) {
  kk::BpSpec S;
  const int rc = kk::sirt_update_spec(S, plan, planes, n_angles, rows, cols, x,
                                      shape, xs, C, cs, mask, ms, lo, hi,
                                      clip_lo, clip_hi, nullptr, 0,
                                      output_scale);
  if (rc != KK_OK) return rc;
  return launch_bp_planes(S, static_cast<hipStream_t>(stream));
}

extern "C" int kk_cone_bp(const kk_plan* plan, const float* proj_tex,
                          int32_t n_angles, int32_t rows, int32_t cols,
                          float* vol, const int32_t shape[3],
                          const int64_t vs[3], float output_scale,
                          int32_t additive, void* stream) {
  kk::BpSpec S;
  const int rc = kk::bp_spec(S, plan, proj_tex, n_angles, rows, cols, vol,
                             shape, vs, output_scale, additive);
  if (rc != KK_OK) return rc;
  return launch_bp_spec(S, 8, static_cast<hipStream_t>(stream));
}

extern "C" int kk_sirt_bp_update(const kk_plan* plan, const float* res_tex,
                                 int32_t n_angles, int32_t rows,
                                 int32_t cols, float* x,
                                 const int32_t shape[3], const int64_t xs[3],
                                 const float* C, const int64_t cs[3],
                                 const float* mask, const int64_t ms[3],
                                 float lo, float hi, int32_t clip_lo,
                                 int32_t clip_hi, float* x_tex,
                                 int32_t x_tex_mask, float output_scale,
                                 void* stream) {
  kk::BpSpec S;
  const int rc = kk::sirt_update_spec(S, plan, res_tex, n_angles, rows, cols,
                                      x, shape, xs, C, cs, mask, ms, lo, hi,
                                      clip_lo, clip_hi, x_tex, x_tex_mask,
                                      output_scale);
  if (rc != KK_OK) return rc;
  return launch_bp_spec(S, 8, static_cast<hipStream_t>(stream));
}
