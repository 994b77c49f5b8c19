// Ray-driven (Joseph) cone-beam forward projection for gfx950.
//
// Behaviour follows cone_fp<DIR_X|Y|Z> of the reference
// (kernelkit/cuda/cone_fp.cu:73-207) as launched by
// kernelkit/kernels/cone_fp.py:195-262: for every angle a ray axis a is
// fixed; each ray through a pixel centre is sampled at the centre of every
// slice along a, bilinearly in the two other axes with zero outside the
// volume, and the sum is scaled by sqrt(1 + a1^2 sc1 + a2^2 sc2) * oscale.
//
// MI355X design:
// * one launch covers all angles and all slices (the reference issues one
//   launch per angle group and 16-slice chunk and accumulates in global
//   memory); each output pixel is written exactly once;
// * the volume is read from slice-major frame textures of (value,
//   b-neighbour) float2 pairs with a zero halo (kk_internal.h), so a sample
//   is: one 64-bit add per coordinate, whose high word is the tap index and
//   low word the weight, one minimum into the halo, and ONE 16-byte load for
//   all four taps;
// * sample coordinates are 64-bit fixed point, a1*i + beta to 2^-33 voxel per
//   slice from the middle one: below the weights' float32 rounding, where the
//   reference's float32 running sums grow along the ray;
// * lanes of a wavefront are 32 consecutive detector rows of two neighbouring
//   columns (fp_lanes).  For rotation about z this makes a
//   wave sample consecutive z voxels of the same (x or y) rows, contiguous
//   memory;
// * the slice loop is wave-uniform: it covers the union of the wave's ray
//   supports (samples outside a ray's support clamp into the zero halo), so
//   the slice base address lives in scalar registers and every tap is an
//   SGPR-base load with a 32-bit per-lane offset; it is software-pipelined
//   one slice deep, which hides part of the latency of the texture misses
//   that dominate at 512^3;
// * for a circular orbit the row step has no in-plane component, so the
//   b-coordinate, its tap row and weight are shared by the thread's R rows
//   ("column-coherent" angles, flagged per angle on the host);
// * per-angle parameters are wave-uniform (scalar loads); workgroups are
//   ordered in groups of kGroupAngles consecutive angles x kGroupCols
//   neighbouring column tiles (angle fastest), groups ordered angle group
//   -> column-tile group -> row band, and each group's ids go to one XCD:
//   neighbouring angles and columns read nearly the same texture lines, so
//   its L2 serves them.
#include <algorithm>
#include <cmath>
#include <new>
#include <type_traits>
#include <vector>

#include "kk_internal.h"

namespace {

constexpr int kWave = 64;
// Wavefronts per workgroup: they share one CU's L1 and move through the slices
// nearly in step, so neighbouring columns' taps hit there (200^3 tilted 1.02,
// 1.02 and 1.13 ms with 4, 8 and 16, 300^3 3.15, 3.28 and 3.63 ms).
constexpr int kColsSingle = 4;
constexpr int kColsBatch = 4;
// The workgroups of kGroupAngles consecutive angles x kGroupCols (single
// problems; kGroupColsBatch in batches) neighbouring column tiles go to
// one XCD together: an XCD holds 256 workgroups of 256 threads (32 CUs x 8).
// Measured on MI355X, 300^3 tilted: 2.98 ms with 16 x 32, 3.06 with 16 x 16,
// 3.12 with 8 x 32, 3.21 with 8 x 16, 4.15 with 4 x 32.  These
// are upper bounds: a group size is the one in [ceil(cap / 2), cap] that
// pads the angles or column tiles least (group_size).
constexpr int32_t kGroupAngles = 16;
constexpr int32_t kGroupCols = 32;
constexpr int32_t kGroupColsBatch = 16;

// Group size for n items, at most cap: the g in [ceil(cap / 2), cap] whose
// whole groups pad n least (the larger g on ties), or n if n <= cap.  Padded
// ids return at once, but the groups go to the XCDs whole, so an XCD dealt
// mostly padded groups idles while others work (160 detector columns = 10
// tiles in groups of 8: about a fifth more time at 128^3 / 180 angles than
// groups of 5).
int32_t group_size(int32_t n, int32_t cap) {
  if (n <= cap) return n;
  int32_t best = cap;
  int64_t best_pad = -1;
  for (int32_t g = cap; g >= (cap + 1) / 2; --g) {
    const int64_t pad = int64_t((n + g - 1) / g) * g - n;
    if (best_pad < 0 || pad < best_pad) {
      best = g;
      best_pad = pad;
    }
  }
  return best;
}

struct FpArgs {
  const char* tex;  // frame textures (byte base)
  float* out;
  // if non-null: the output base is out_ptrs[index along logical axis
  // ptr_axis] instead of out (whose stride along that axis is then 0)
  const int64_t* out_ptrs;
  int32_t ptr_axis;
  int64_t os0, os1, os2;  // output strides: angle, row, col
  int64_t out_dual;       // if nonzero: also write out[o + out_dual]
  const float* y;         // mode 2: measured projections
  int64_t ys0, ys1, ys2;
  const float* R;  // mode 2: ray weights
  int64_t rs0, rs1, rs2;
  int32_t rows, cols, n_angles;
  int32_t row_tiles, col_tiles;
  int32_t row_shift;  // a wavefront is 2^row_shift rows x 64 >> row_shift cols
  int32_t mode;  // 0: out = p, 1: out += p, 2: out = (p - y) * R
  int32_t xcd_group;
  // workgroup groups: grp_a angles x grp_c column tiles (ids past the
  // angles or column tiles, which pad the grid to whole groups, return)
  int32_t grp_a, grp_c;
  int64_t total_blocks;
};

// Narrow [lo, hi] (slice indices, initially [0, n_a - 1]) to the slices i
// with 0 < a*i + beta < n + 1 (padded coordinates).  For slopes below 1e-3
// the division is not trusted; the ray is then only dropped when it stays
// outside over the whole slice range.  Over-inclusion is harmless: clamped
// samples outside the volume read the zero halo.
__device__ __forceinline__ void clip_range(float a, float beta, float n1,
                                           float last, float& lo,
                                           float& hi) {
  if (fabsf(a) < 1e-3f) {
    const float e0 = beta, e1 = fmaf(a, last, beta);
    if (fmaxf(e0, e1) <= 0.f || fminf(e0, e1) >= n1) {
      lo = 3e38f;
      hi = -3e38f;
    }
    return;
  }
  const float inv = 1.f / a;
  const float t0 = (0.f - beta) * inv;
  const float t1 = (n1 - beta) * inv;
  lo = fmaxf(lo, fminf(t0, t1));
  hi = fminf(hi, fmaxf(t0, t1));
}

// Bilinear value from the 16-byte tap record (v[b][c], v[b+1][c],
// v[b][c+1], v[b+1][c+1]): lerp along b, then along c.
__device__ __forceinline__ float bilerp(kk_float4u t, float fb, float fc) {
  const float l0 = fmaf(fb, t.y - t.x, t.x);
  const float l1 = fmaf(fb, t.w - t.z, t.z);
  return fmaf(fc, l1 - l0, l0);
}

// The four taps and two weights of one slice for the R rays of a thread.
template <int R, int NB>
struct SliceTaps {
  kk_float4u t[R];
  float fb[NB];
  float fc[R];
};

// x as 64-bit fixed point with 32 fraction bits (|x| < 2^31).
__device__ __forceinline__ int64_t to_fixed(double x) {
  const double fl = floor(x);
  const uint32_t lo = static_cast<uint32_t>(
      fmin(fma(x - fl, 4294967296.0, 0.5), 4294967295.0));
  return static_cast<int64_t>(
      (static_cast<uint64_t>(static_cast<uint32_t>(static_cast<int32_t>(fl)))
       << 32) |
      lo);
}

// Coordinates of a thread's R rays at a slice, and their steps per slice, as
// 64-bit fixed point (to_fixed): the high word is the padded element, the low
// word the weight.  NB = 1: the b coordinate is shared by the R rays (column-
// coherent angles).  Coordinates outside the volume (below the halo: a
// negative element, huge as unsigned) go to element n + 1, whose taps are all
// halo zeros whatever the weight: one unsigned minimum.
//
// (A sample took float64 coordinates before, their clamps or a second pass for
// the slices that lie inside for a whole wavefront: 27 vector instructions a
// gather, now 22.  200^3 tilted 1.40 -> 1.00 ms together with fp_lanes, 300^3
// 4.83 -> 3.0 ms, 400^3 / 200 wobbling angles 10.3 -> 8.0 ms, 64^3 58 -> 46 us.
// The address units are busy in 87% of the cycles at 256^3 / 360 wobbling angles,
// misses included (16 cycles a gather by themselves); a deeper pipeline was
// slower, so what is left is the L2's latency and the L1's misses.)
template <int R, int NB>
struct RayWalk {
  int64_t b[NB], c[R];
  int64_t gb[NB], gc[R];
};

// Slices walked from one float64 coordinate, at most: a step's rounding (2^-33
// voxel) then adds up to 512 of them, 2^-24 voxel, like a weight's own float32
// rounding, however long the volume's axis is.
constexpr int32_t kSegment = 1024;

// Coordinate a i + b at slice mid, the middle of the slices that the ray
// meets, and its step: the step's rounding (2^-33 voxel per slice) adds up over
// half of them at most, and cancels in the ray's sum (a ray that only grazes
// the volume, whose sum a reconstruction divides by, loses no accuracy).
// A ray nearly parallel to the slices, whose coordinates leave the fixed-point
// range, is inside the volume (n1 - 1 voxels) at one slice at most: it has its
// coordinate there, and at the others one outside.
__device__ __forceinline__ void fixed_ray(double a, double b, int32_t na,
                                          int32_t mid, float n1, int64_t& at,
                                          int64_t& step) {
  constexpr double kRange = 1073741824.0;  // 2^30
  double g = a, x = fma(a, static_cast<double>(mid), b);
  int32_t far = 0;
  if (!(fabs(a) * static_cast<double>(na) + fabs(b) < kRange)) {
    const double r = __builtin_amdgcn_rcp(a);
    const double i = rint(fmin(
        fmax((0.5 * n1 - b) * fma(r, fma(-a, r, 1.0), r), 0.0), na - 1.0));
    x = fmin(fmax(fma(a, i, b), -kRange), kRange);
    g = copysign(kRange / 2 / static_cast<double>(na), a);
    far = mid - static_cast<int32_t>(i);
  }
  step = to_fixed(g);
  at = to_fixed(x) + static_cast<int64_t>(far) * step;
}

__device__ __forceinline__ void split_fixed(int64_t x, uint32_t n1,
                                            uint32_t& idx, float& frac) {
  const uint64_t u = static_cast<uint64_t>(x);
  idx = min(static_cast<uint32_t>(u >> 32), n1);
  frac = static_cast<float>(static_cast<uint32_t>(u)) * 0x1p-32f;
}

// Weights and tap loads of one slice for R rays; the walk moves on to the
// next.
template <int R, int NB>
__device__ __forceinline__ void fetch_slice(const char* __restrict__ slice,
                                            uint32_t sbb, uint32_t nb1,
                                            uint32_t nc1, RayWalk<R, NB>& w,
                                            SliceTaps<R, NB>& s) {
  uint32_t ob = 0;
#pragma unroll
  for (int k = 0; k < R; ++k) {
    if (k < NB) {
      uint32_t ib;
      split_fixed(w.b[k], nb1, ib, s.fb[k]);
      ob = __umul24(ib, sbb);
      // one multiply for the R rays (not a multiply-add per ray)
      if constexpr (NB == 1) asm volatile("" : "+v"(ob));
      w.b[k] += w.gb[k];
      asm volatile("" : "+v"(w.b[k]));
    }
    uint32_t ic;
    split_fixed(w.c[k], nc1, ic, s.fc[k]);
    w.c[k] += w.gc[k];
    // (coordinates stay one register pair each, stepped: the optimizer would
    // split them into words and multiples of the step)
    asm volatile("" : "+v"(w.c[k]));
    s.t[k] = kk_ld4(slice, ob + (ic << 3));
  }
}

template <int R, int NB>
__device__ __forceinline__ void add_slice(const SliceTaps<R, NB>& s,
                                          float (&acc)[R]) {
#pragma unroll
  for (int k = 0; k < R; ++k)
    acc[k] += bilerp(s.t[k], s.fb[NB == 1 ? 0 : k], s.fc[k]);
}

// Trace slices [i0, i1] (wave-uniform) for R rays of a thread from their
// coordinates at i0.  PIPE software-pipelines the pass: the taps of slice
// i + 1 are requested before slice i is interpolated, so a wavefront keeps two
// slices of gathers in flight (two register buffers, the loop unrolled by
// two so that they swap roles without copies; the request past i1 repeats
// slice i1 and is discarded).  The scheduling barriers keep each request
// ahead of the interpolation (the scheduler would otherwise sink the loads
// next to their use).  Measured on MI355X at 512^3 / 720 angles: 5% faster
// than one slice in flight; three slices in flight (at 6 instead of 8
// wavefronts per SIMD, for the registers) are no faster than two.
template <int R, int NB, bool PIPE>
__device__ __forceinline__ void trace(const kk::FpAngle& P,
                                      const char* __restrict__ frame,
                                      RayWalk<R, NB>& w, int32_t i0,
                                      int32_t i1, float (&acc)[R]) {
  const uint32_t nb1 = static_cast<uint32_t>(P.nb) + 1;
  const uint32_t nc1 = static_cast<uint32_t>(P.nc) + 1;
  const uint32_t sab = P.sab, sbb = P.sbb;
  auto fetch = [&](int32_t i, SliceTaps<R, NB>& s) {
    fetch_slice<R, NB>(frame + static_cast<size_t>(min(i, i1)) * sab, sbb,
                       nb1, nc1, w, s);
  };
  if constexpr (!PIPE) {
    for (int32_t i = i0; i <= i1; ++i) {
      SliceTaps<R, NB> A;
      fetch(i, A);
      add_slice(A, acc);
    }
  } else {
    SliceTaps<R, NB> A, B;
    int32_t i = i0;
    if ((i1 - i0) % 2 == 0) {
      fetch(i, A);
      add_slice(A, acc);
      if (++i > i1) return;
    }
    fetch(i, A);
    for (; i < i1; i += 2) {
      fetch(i + 1, B);
      __builtin_amdgcn_sched_barrier(0);
      add_slice(A, acc);
      fetch(i + 2, A);
      __builtin_amdgcn_sched_barrier(0);
      add_slice(B, acc);
    }
  }
}

// Rays that graze the volume.  The fixed-point coordinates are good to ~1e-10
// voxel, the weights made of them to 1e-10 of a voxel's value: less than their
// float32 rounding except right at the low faces (padded coordinates just above
// 0), where a float64 coordinate gives a weight of 24 good bits however small it
// is.  A reconstruction divides by the sums of weights, so rays that nowhere
// reach deeper than kGraze into the volume are traced again in float64, over
// their own few slices.
constexpr float kGraze = 0x1p-6f;

// Narrows [lo, hi] to the slices where a i + b lies in [0, n1] (to 1e-3 voxel
// too many) and [dlo, dhi] to those where it is at least kGraze.
__device__ __forceinline__ void graze_range(float a, float b, float n1,
                                            float& lo, float& hi, float& dlo,
                                            float& dhi) {
  const float inv = 1.f / (fabsf(a) > 1e-7f ? a : 1e-7f);
  const float t = -b * inv, g = kGraze * inv, w = n1 * inv;
  const float e = 1e-3f * fabsf(inv);
  lo = fmaxf(lo, fminf(t, t + w) - e);
  hi = fminf(hi, fmaxf(t, t + w) + e);
  dlo = fmaxf(dlo, fminf(t + g, t + w));
  dhi = fminf(dhi, fmaxf(t + g, t + w));
}
__device__ __forceinline__ bool grazes(double a1, double b1, double a2,
                                       double b2, float nb1, float nc1,
                                       float last, float& lo, float& hi) {
  float dlo = 0.f, dhi = last;
  lo = 0.f;
  hi = last;
  graze_range(static_cast<float>(a1), static_cast<float>(b1), nb1, lo, hi,
              dlo, dhi);
  graze_range(static_cast<float>(a2), static_cast<float>(b2), nc1, lo, hi,
              dlo, dhi);
  lo = ceilf(lo);
  hi = floorf(hi);
  return lo <= hi && !(ceilf(dlo) <= floorf(dhi));
}

// The sum of ray (row, col) if it grazes the volume.  taps(i, ib, ic) are the
// four values at padded element (ib, ic) of slice i.
template <class Taps>
__device__ __forceinline__ bool graze_sum(const kk::FpAngle& P, int32_t row,
                                          int32_t col, float& sum,
                                          Taps taps) {
  double a1, b1, a2, b2;
  float lo, hi;
  if (!kk_fp_ray(P, row, col, a1, b1, a2, b2) ||
      !grazes(a1, b1, a2, b2, static_cast<float>(P.nb + 1),
              static_cast<float>(P.nc + 1), static_cast<float>(P.na - 1), lo,
              hi))
    return false;
  const double nb1 = static_cast<double>(P.nb + 1);
  const double nc1 = static_cast<double>(P.nc + 1);
  sum = 0.f;
  for (int32_t i = static_cast<int32_t>(lo); i <= static_cast<int32_t>(hi);
       ++i) {
    const double fi = static_cast<double>(i);
    uint32_t ib, ic;
    float fb, fc;
    kk_fp_coord(a1, b1, fi, nb1, ib, fb);
    kk_fp_coord(a2, b2, fi, nc1, ic, fc);
    sum += bilerp(taps(i, ib, ic), fb, fc);
  }
  return true;
}

// One workgroup's tile (row band rt, angle, column tile ct) of logical
// block id `bid`.  ALL_COLC: every angle of the launch is column-coherent,
// so a thread keeps one b slope/intercept for its R rays (fewer registers,
// more wavefronts in flight); otherwise the angle's flag picks the path.
// FAR: the plan has an axis of more than kSegment slices.
template <int R, bool ALL_COLC, bool PIPE, int COLS, bool FAR,
          bool PTRS = false>
__device__ __forceinline__ void fp_tile_at(
    const kk::FpAngle* __restrict__ tab, int32_t ti, const FpArgs& A,
    int32_t ang, int32_t ct, int32_t rt) {
  constexpr int NB = ALL_COLC ? 1 : R;
  const int32_t lane = int32_t(threadIdx.x) & (kWave - 1);
  const int32_t rows = 1 << A.row_shift;  // of a wavefront
  const int32_t col =
      ((ct * COLS + int32_t(threadIdx.x) / kWave) << (6 - A.row_shift)) +
      (lane >> A.row_shift);
  const int32_t row0 = rt * (rows * R) + (lane & (rows - 1));

  const kk::FpAngle& P = tab[ti];
  const float nb1 = static_cast<float>(P.nb + 1);
  const float nc1 = static_cast<float>(P.nc + 1);
  const float last = static_cast<float>(P.na - 1);

  RayWalk<R, NB> w;
  float wscale[R];
  int32_t ilo = 0x7fffffff, ihi = -1;
  int32_t mb[NB], mc[R];  // slices of the coordinates in w
  bool graze = false;
#pragma unroll
  for (int k = 0; k < R; ++k) {
    const int32_t row = row0 + rows * k;
    // rays outside the detector, or parallel to the slices, contribute
    // nothing: they are parked at padded coordinate 1 with weight 0 (for
    // column-coherent angles the b part of every ray of the thread equals
    // that of its first ray)
    double a1, b1, a2, b2;
    const bool ok = row < A.rows && col < A.cols &&
                    kk_fp_ray(P, row, col, a1, b1, a2, b2);
    wscale[k] = ok ? kk_fp_weight(P, a1, a2) : 0.f;
    a1 = ok ? a1 : 0.0;
    b1 = ok ? b1 : 1.0;
    a2 = ok ? a2 : 0.0;
    b2 = ok ? b2 : 1.0;
    float lo = 0.f, hi = last;
    clip_range(static_cast<float>(a1), static_cast<float>(b1), nb1, last, lo,
               hi);
    const float lob = lo, hib = hi;
    clip_range(static_cast<float>(a2), static_cast<float>(b2), nc1, last, lo,
               hi);
    float glo, ghi;
    graze = graze || (ok && grazes(a1, b1, a2, b2, nb1, nc1, last, glo, ghi));
    auto middle = [&](float l, float h) {
      return static_cast<int32_t>(fminf(fmaxf(0.5f * (l + h), 0.f), last));
    };
    const int32_t mid = middle(lo, hi);
    if (k < NB) {
      // column-coherent angles: the column's own middle, so that rays have
      // the same bits whichever rays share their b coordinate
      mb[k] = P.colc ? middle(lob, hib) : mid;
      fixed_ray(a1, b1, P.na, mb[k], nb1, w.b[k], w.gb[k]);
    }
    mc[k] = mid;
    fixed_ray(a2, b2, P.na, mid, nc1, w.c[k], w.gc[k]);
    if (ok && lo <= hi + 2.f) {
      ilo = min(ilo, max(0, static_cast<int32_t>(floorf(lo)) - 1));
      ihi = max(ihi, min(P.na - 1, static_cast<int32_t>(ceilf(hi)) + 1));
    }
  }
  ilo = kk_wave_min(ilo);
  ihi = kk_wave_max(ihi);

  float acc[R];
#pragma unroll
  for (int k = 0; k < R; ++k) acc[k] = 0.f;
  if (ilo <= ihi) {
#pragma unroll
    for (int k = 0; k < NB; ++k)
      w.b[k] += static_cast<int64_t>(ilo - mb[k]) * w.gb[k];
#pragma unroll
    for (int k = 0; k < R; ++k)
      w.c[k] += static_cast<int64_t>(ilo - mc[k]) * w.gc[k];
    const char* frame = A.tex + P.tex_off;
    if constexpr (!FAR) {
      trace<R, NB, PIPE>(P, frame, w, ilo, ihi, acc);
    } else {
#pragma unroll 1
      for (int32_t s = ilo; s <= ihi; s += kSegment) {
        const int32_t e = min(ihi, s + kSegment - 1), mid = s + (e - s) / 2;
#pragma unroll
        for (int k = 0; k < R; ++k) {
          const int32_t row = row0 + rows * k;
          double a1, b1, a2, b2;
          if (!(row < A.rows && col < A.cols &&
                kk_fp_ray(P, row, col, a1, b1, a2, b2))) {
            a1 = a2 = 0.0;
            b1 = b2 = 1.0;
          }
          if (k < NB) {
            fixed_ray(a1, b1, P.na, mid, nb1, w.b[k], w.gb[k]);
            w.b[k] -= static_cast<int64_t>(mid - s) * w.gb[k];
          }
          fixed_ray(a2, b2, P.na, mid, nc1, w.c[k], w.gc[k]);
          w.c[k] -= static_cast<int64_t>(mid - s) * w.gc[k];
        }
        trace<R, NB, PIPE>(P, frame, w, s, e, acc);
      }
    }
    if (graze) {
#pragma unroll 1
      for (int32_t k = 0; k < R; ++k) {
        float v;
        if (row0 + rows * k < A.rows &&
            graze_sum(P, row0 + rows * k, col, v,
                      [&](int32_t i, uint32_t ib, uint32_t ic) {
                        return kk_ld4(frame + static_cast<size_t>(i) * P.sab,
                                      __umul24(ib, P.sbb) + (ic << 3));
                      })) {
#pragma unroll
          for (int t = 0; t < R; ++t) acc[t] = t == k ? v : acc[t];
        }
      }
    }
  }

#pragma unroll
  for (int k = 0; k < R; ++k) {
    const int32_t row = row0 + rows * k;
    if (row >= A.rows || col >= A.cols) continue;
    float val = acc[k] * wscale[k];
    const int64_t o = ang * A.os0 + row * A.os1 + col * A.os2;
    float* out = A.out;
    if constexpr (PTRS)
      out = reinterpret_cast<float*>(
          A.out_ptrs[A.ptr_axis == 0 ? ang : (A.ptr_axis == 1 ? row : col)]);
    if (A.mode == 1) {
      out[o] += val;
      continue;
    }
    if (A.mode == 2) {
      const float yv = A.y[ang * A.ys0 + row * A.ys1 + col * A.ys2];
      const float rv = A.R[ang * A.rs0 + row * A.rs1 + col * A.rs2];
      val = (val - yv) * rv;
    }
    out[o] = val;
    if (A.out_dual) out[o + A.out_dual] = val;
  }
}

// Decode logical block id `bid` (groups of grp_a angles x grp_c column
// tiles, angle fastest inside a group; groups ordered angle group, then
// column-tile group, then row band); false for the grid's padding.
__device__ __forceinline__ bool fp_decode(const FpArgs& A, int64_t bid,
                                          int32_t& ang, int32_t& ct,
                                          int32_t& rt) {
  const int32_t ga = A.grp_a, gc = A.grp_c;
  const int64_t inner = bid % (int64_t(ga) * gc);
  const int64_t outer = bid / (int64_t(ga) * gc);
  const int32_t nag = (A.n_angles + ga - 1) / ga;
  const int32_t ncg = (A.col_tiles + gc - 1) / gc;
  ang = static_cast<int32_t>(outer % nag) * ga +
        static_cast<int32_t>(inner % ga);
  const int64_t t = outer / nag;
  ct = static_cast<int32_t>(t % ncg) * gc + static_cast<int32_t>(inner / ga);
  rt = static_cast<int32_t>(t / ncg);
  return ang < A.n_angles && ct < A.col_tiles;
}

// Trace the tile of logical block id `bid`.  TABLE_IN_MEMORY: the angle
// table pointer was read from a descriptor (batch kernels); the record is
// then copied through constant-memory (scalar) loads first.  A table passed
// as a kernel argument is read in place (the compiler scalarizes it by
// itself; the explicit copy measured 5% slower at 512^3 / 720 angles).
template <int R, bool ALL_COLC, bool PIPE, int COLS, bool TABLE_IN_MEMORY,
          bool FAR, bool PTRS = false>
__device__ __forceinline__ void fp_tile(const kk::FpAngle* __restrict__ tab,
                                        const FpArgs& A, int64_t bid) {
  int32_t ang, ct, rt;
  if (!fp_decode(A, bid, ang, ct, rt)) return;
  if constexpr (TABLE_IN_MEMORY) {
    const kk::FpAngle rec = kk_uniform_load(tab + ang);
    fp_tile_at<R, ALL_COLC, PIPE, COLS, FAR, PTRS>(&rec, 0, A, ang, ct, rt);
  } else {
    fp_tile_at<R, ALL_COLC, PIPE, COLS, FAR, PTRS>(tab, ang, A, ang, ct, rt);
  }
}

// Wavefronts per SIMD (register caps): 8 up to two rows per thread, 5 at
// four.
constexpr int fp_waves(int r) { return r <= 2 ? 8 : 5; }
// Slice pipelining: with one row per thread (200^3 tilted 1.06 ms, without
// 1.25; with two rows 1.30 and 1.18).
constexpr bool fp_pipe(int r) { return r <= 1; }

// One row per thread: whether the angles are column-coherent is the same.
// PTRS: output through the table of entry pointers (kk_cone_fp_ptrs); a
// separate instantiation, so the plain kernel's code is unchanged.
template <bool FAR, bool PTRS>
__global__ __launch_bounds__(kColsSingle * kWave, fp_waves(1)) void
cone_fp_kernel(const kk::FpAngle* __restrict__ tab, FpArgs A) {
  fp_tile<1, false, fp_pipe(1), kColsSingle, false, FAR, PTRS>(
      tab, A, kk_xcd_remap(blockIdx.x, A.total_blocks, A.xcd_group));
}


// ---- column-coherent launches: one volume line per column and slice ------
//
// When every angle is column-coherent (circular orbits), the rays of one
// detector column meet a slice at one b coordinate: all of its samples there
// interpolate between the same two volume rows, at c coordinates affine in
// the detector row.  A wavefront owns 64 R consecutive rows of one column.
// Per slice it reads the window of the two rows that its rays reach (one
// coalesced 4-byte load per 64 elements and row, from planes: the volume as
// plain floats), interpolates them along b once per element, keeps that line
// in its own LDS words, and every ray reads two neighbouring words of it.
// The arithmetic per sample is bilerp's (along b, then along c).
//
// What bounds it (MI355X): a 16-byte gather costs a CU 16 cycles per 64
// samples whatever its pattern, a coalesced 4-byte load 4.5, an LDS store
// 5.2 and a paired LDS read at neighbouring addresses 5.0; so with windows
// of W x 64 elements a sample costs 9 W / R cycles of loads beside
// (5.2 W + 5 R) / R of LDS and ~9 of vector instructions.  Measured: FP
// 512^3 / 720 x 768^2 85.7-91 -> 57 ms, 128^3 / 180 x 160^2 0.43 -> 0.27 ms
// (R = 1, 2, 3, 4 at the former: 141, 91, 64, 57 ms).  Of the 57 ms, 37
// remain without the loads and 47 when every load hits the L2: what is left
// is vector issue first, then misses (a second slice in flight, two columns
// per wavefront and slabs of slices were no faster).
//
// c coordinates are 64-bit fixed point (32 fraction bits), stepped by one
// 64-bit add per slice: the high word is the element, the low word the
// weight.  Their error (the slope's rounding, 2^-33 voxel per slice from the
// middle one) stays at the weights' own float32 rounding for the volumes that
// line_spacing admits.
// Columns (wavefronts) per workgroup.  They walk the same slices behind one
// barrier per slice, so that neighbouring columns' rows meet in the CU's L1
// (57.0 ms against 62.5 without; 8 and 16 columns 59.2 and 61.9 ms).
constexpr int kLineWaves = 4;
constexpr int32_t kLineGroupAngles = 8;   // workgroup groups, as kGroupAngles
constexpr int32_t kLineGroupCols = 32;    // (16 x 16: 58.7 ms)
constexpr int kLineChunks = 4;                  // windows up to 4 x 64
constexpr int kLineWords = 64 * kLineChunks;    // LDS words per wavefront
constexpr int64_t kLineEps = int64_t(1) << 18;  // 2^-14 voxel, fixed point

__device__ __forceinline__ int64_t bcast64(int64_t v, int32_t lane) {
  const uint32_t lo = static_cast<uint32_t>(__builtin_amdgcn_readlane(
      static_cast<int32_t>(static_cast<uint64_t>(v)), lane));
  const uint32_t hi = static_cast<uint32_t>(__builtin_amdgcn_readlane(
      static_cast<int32_t>(static_cast<uint64_t>(v) >> 32), lane));
  return static_cast<int64_t>((static_cast<uint64_t>(hi) << 32) | lo);
}

__device__ __forceinline__ int32_t fixed_int(int64_t x) {
  return static_cast<int32_t>(static_cast<uint64_t>(x) >> 32);
}
__device__ __forceinline__ float fixed_frac(int64_t x) {
  return static_cast<float>(static_cast<uint32_t>(x)) * 0x1p-32f;
}

// A wave's state along the slices: per-lane c coordinates and steps of its R
// rays, wave-uniform b coordinate and window start with their steps.
template <int R>
struct LineWalk {
  int64_t X[R], S[R];
  int64_t B, SB, E, SE;
};

// n slices from `slice` (byte address of the plane) with windows of W chunks.
// The next slice's loads are in flight while a slice is interpolated.
template <int R, int W>
__device__ __forceinline__ void line_trace(LineWalk<R>& w, int32_t n,
                                           const char*& slice, uint64_t sab,
                                           uint32_t sbb, int32_t row_bytes,
                                           int32_t nb1, uint32_t line_at,
                                           uint32_t lane4, float (&acc)[R]) {
  typedef __attribute__((address_space(3))) float* lds_ptr;
  if (n <= 0) return;
  float v0[W], v1[W], fb;
  int32_t z0;
  // Both rows' window at the current slice, through buffer descriptors that
  // hold one row each: elements before the row (negative offsets, i.e. large
  // unsigned ones) and after it read as zero.
  auto request = [&]() {
    const int32_t jb = fixed_int(w.B);
    const int32_t j = min(max(jb, 0), nb1);
    fb = fixed_frac(j == jb ? w.B : 0);
    z0 = __builtin_amdgcn_readfirstlane(fixed_int(w.E));
    const char* row = slice + static_cast<uint64_t>(
        static_cast<uint32_t>(j) * sbb);
    const auto r0 = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<char*>(row), 0, row_bytes, 0x00020000);
    const auto r1 = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<char*>(row + sbb), 0, row_bytes, 0x00020000);
#pragma unroll
    for (int c = 0; c < W; ++c) {
      // (in asm, so that no negative offset meets an immediate)
      uint32_t o;
      asm("v_add_u32 %0, %1, %2"
          : "=v"(o)
          : "s"((z0 + c * kWave) * 4), "v"(lane4));
      v0[c] = __builtin_bit_cast(
          float, __builtin_amdgcn_raw_buffer_load_b32(r0, o, 0, 0));
      v1[c] = __builtin_bit_cast(
          float, __builtin_amdgcn_raw_buffer_load_b32(r1, o, 0, 0));
    }
    w.B += w.SB;
    w.E += w.SE;
    slice += sab;
  };
  const lds_ptr st = (lds_ptr)(line_at + lane4);
  request();
  for (;;) {
    __builtin_amdgcn_s_barrier();
#pragma unroll
    for (int c = 0; c < W; ++c)
      st[c * kWave] = fmaf(fb, v1[c] - v0[c], v0[c]);
    __builtin_amdgcn_wave_barrier();
    const uint32_t at = line_at - static_cast<uint32_t>(z0) * 4u;
    float l0[R], l1[R];
#pragma unroll
    for (int k = 0; k < R; ++k) {
      uint32_t q;  // one shift-add of the element (not a 64-bit shift)
      asm("v_lshl_add_u32 %0, %1, 2, %2"
          : "=v"(q)
          : "v"(fixed_int(w.X[k])), "s"(at));
      l0[k] = ((lds_ptr)q)[0];
      l1[k] = ((lds_ptr)q)[1];
    }
    const bool more = --n > 0;
    if (more) request();
#pragma unroll
    for (int k = 0; k < R; ++k) {
      acc[k] += fmaf(fixed_frac(w.X[k]), l1[k] - l0[k], l0[k]);
      w.X[k] += w.S[k];
    }
    if (!more) break;
  }
}

template <int R, bool PTRS>
__global__ __launch_bounds__(kLineWaves * kWave, 8) void cone_fp_line_kernel(
    const kk::FpAngle* __restrict__ tab, FpArgs A) {
  __shared__ float lines[kLineWaves * kLineWords];
  int32_t ang, ct, rt;
  if (!fp_decode(A, kk_xcd_remap(blockIdx.x, A.total_blocks, A.xcd_group),
                 ang, ct, rt))
    return;
  const int32_t lane = int32_t(threadIdx.x) & (kWave - 1);
  const int32_t wave = __builtin_amdgcn_readfirstlane(
      int32_t(threadIdx.x) / kWave);
  // columns past the detector repeat the last one (not written out)
  const int32_t wcol = ct * kLineWaves + wave;
  const int32_t col = min(wcol, A.cols - 1);
  const int32_t row0 = rt * (kWave * R);
  const kk::FpAngle& P = tab[ang];
  const float nb1 = static_cast<float>(P.nb + 1);
  const float nc1 = static_cast<float>(P.nc + 1);
  const float last = static_cast<float>(P.na - 1);

  double a1 = 0.0, b1 = 0.0, a2[R], b2[R];
  int32_t ilo = 0x7fffffff, ihi = -1;
  bool graze = false;
#pragma unroll
  for (int k = 0; k < R; ++k) {
    // rows past the detector repeat the last one (not written out)
    const int32_t row = min(row0 + kWave * k + lane, A.rows - 1);
    // (no ray is parallel to the slices: line_spacing)
    kk_fp_ray(P, row, col, a1, b1, a2[k], b2[k]);
    float lo, hi;
    graze = graze || grazes(a1, b1, a2[k], b2[k], nb1, nc1, last, lo, hi);
    lo = 0.f, hi = last;
    clip_range(static_cast<float>(a1), static_cast<float>(b1), nb1, last, lo,
               hi);
    clip_range(static_cast<float>(a2[k]), static_cast<float>(b2[k]), nc1, last,
               lo, hi);
    if (lo <= hi + 2.f) {
      ilo = min(ilo, max(0, static_cast<int32_t>(floorf(lo)) - 1));
      ihi = max(ihi, min(P.na - 1, static_cast<int32_t>(ceilf(hi)) + 1));
    }
  }
  {
    __shared__ int32_t lim[2][16];
    lim[0][wave] = kk_wave_min(ilo);
    lim[1][wave] = kk_wave_max(ihi);
    __syncthreads();
    #pragma unroll
    for (int32_t t = 0; t < kLineWaves; ++t) {
      ilo = min(ilo, lim[0][t]);
      ihi = max(ihi, lim[1][t]);
    }
  }
  ilo = __builtin_amdgcn_readfirstlane(ilo);
  ihi = __builtin_amdgcn_readfirstlane(ihi);

  float acc[R];
#pragma unroll
  for (int k = 0; k < R; ++k) acc[k] = 0.f;
  if (ilo <= ihi) {
    // from the middle slice, where the steps' rounding cancels
    const int32_t n = ihi - ilo + 1;
    const double fm = static_cast<double>(ilo + n / 2);
    LineWalk<R> w;
#pragma unroll
    for (int k = 0; k < R; ++k) {
      w.S[k] = to_fixed(a2[k]);
      w.X[k] = to_fixed(fma(a2[k], fm, b2[k])) -
               static_cast<int64_t>(n / 2) * w.S[k];
    }
    w.SB = bcast64(to_fixed(a1), 0);
    w.B = bcast64(to_fixed(fma(a1, fm, b1)), 0) -
          static_cast<int64_t>(n / 2) * w.SB;
    // the window lies between the c coordinates of the first and last rows
    // (those between lie between up to the rounding that kLineEps covers);
    // which is the lower does not change along the slices
    const int64_t E0 = bcast64(w.X[0], 0), E1 = bcast64(w.X[R - 1], kWave - 1);
    const int64_t S0 = bcast64(w.S[0], 0), S1 = bcast64(w.S[R - 1], kWave - 1);
    const bool up = E1 + (n >> 1) * S1 >= E0 + (n >> 1) * S0;
    w.E = bcast64((up ? E0 : E1) - kLineEps, 0);
    w.SE = bcast64(up ? S0 : S1, 0);
    // window widths (elements) at the first and the last slice, linear
    // between; one chunk fewer where the window is that narrow
    const float d0 = static_cast<float>(up ? E1 - E0 : E0 - E1) * 0x1p-32f;
    const float ds = static_cast<float>(up ? S1 - S0 : S0 - S1) * 0x1p-32f;
    const float wa = d0 + 3.1f, wb = fmaf(ds, static_cast<float>(n - 1), wa);
    const int32_t top = __builtin_amdgcn_readfirstlane(
        static_cast<int32_t>(ceilf(fmaxf(wa, wb) * (1.f / kWave))));
    const float fit = static_cast<float>((top - 1) * kWave);
    int32_t na = 0, nb = 0;  // narrow slices at the start / at the end
    if (fmaxf(wa, wb) <= fit) na = n;
    else if (wa <= fit && ds > 0.f)
      na = min(n, max(0, static_cast<int32_t>((fit - wa) / ds)));
    else if (wb <= fit && ds < 0.f)
      nb = min(n, max(0, static_cast<int32_t>((fit - wb) / -ds)));
    na = __builtin_amdgcn_readfirstlane(na);
    nb = __builtin_amdgcn_readfirstlane(nb);

    const uint32_t sbb = static_cast<uint32_t>(P.nc + kk::kHalo) * 4u;
    const uint64_t sab = static_cast<uint64_t>(P.nb + kk::kHalo) * sbb;
    const char* slice = A.tex + (P.tex_off >> 1) +
                        static_cast<uint64_t>(ilo) * sab;
    typedef __attribute__((address_space(3))) float* lds_ptr;
    const uint32_t line_at = __builtin_amdgcn_readfirstlane(
        static_cast<uint32_t>(reinterpret_cast<uintptr_t>(
            (lds_ptr)(lines + wave * kLineWords))));
    const uint32_t lane4 = static_cast<uint32_t>(lane) * 4u;
    const int32_t row_bytes = static_cast<int32_t>(sbb);
#pragma unroll 1
    for (int32_t pass = 0; pass < 3; ++pass) {
      const int32_t m = pass == 0 ? na : (pass == 1 ? n - na - nb : nb);
      const int32_t chunks = pass == 1 ? top : top - 1;
      if (m <= 0) continue;
#define KK_LINE(W_)                                                        \
  line_trace<R, W_>(w, m, slice, sab, sbb, row_bytes, P.nb + 1, line_at, \
                    lane4, acc)
      if (chunks <= 1) KK_LINE(1);
      else if (chunks == 2) KK_LINE(2);
      else if (chunks == 3) KK_LINE(3);
      else KK_LINE(4);
#undef KK_LINE
    }
  }
  if (graze) {
    const uint32_t sbb = static_cast<uint32_t>(P.nc + kk::kHalo) * 4u;
    const uint64_t sab = static_cast<uint64_t>(P.nb + kk::kHalo) * sbb;
    const char* frame = A.tex + (P.tex_off >> 1);
#pragma unroll 1
    for (int32_t k = 0; k < R; ++k) {
      float x;
      if (graze_sum(P, min(row0 + kWave * k + lane, A.rows - 1), col, x,
                    [&](int32_t i, uint32_t ib, uint32_t ic) {
                      const float* v = reinterpret_cast<const float*>(
                          frame + i * sab + static_cast<uint64_t>(ib) * sbb) +
                          ic;
                      const float* u = v + sbb / 4;
                      return kk_float4u{v[0], u[0], v[1], u[1]};
                    })) {
#pragma unroll
        for (int t = 0; t < R; ++t) acc[t] = t == k ? x : acc[t];
      }
    }
  }
#pragma unroll
  for (int k = 0; k < R; ++k) {
    const int32_t row = row0 + kWave * k + lane;
    if (row >= A.rows || wcol >= A.cols) continue;
    double ra1, rb1, ra2, rb2;
    const float wt = kk_fp_ray(P, row, col, ra1, rb1, ra2, rb2)
                         ? kk_fp_weight(P, ra1, ra2)
                         : 0.f;
    const int64_t o = ang * A.os0 + row * A.os1 + col * A.os2;
    float* out = A.out;
    if constexpr (PTRS)
      out = reinterpret_cast<float*>(
          A.out_ptrs[A.ptr_axis == 0 ? ang : (A.ptr_axis == 1 ? row : col)]);
    if (A.mode == 1)
      out[o] += acc[k] * wt;
    else
      out[o] = acc[k] * wt;
  }
}

}  // namespace

namespace {

// Rows per thread, and rows of a wavefront (2^shift; the other lanes are
// neighbouring columns), where the caller leaves them open.  Single problems:
// one row, wavefronts of 32 x 2.  Measured, 1 row x 64, 1 x 32, 2 x 64, 2 x 32
// and 4 x 16 (139, 213 and 319 rows: 150 x 141 x 93, 200^3 and 300^3 tilted):
// 0.49, 0.45, 0.52, 0.50 and 0.45 ms; 1.05, 1.00, 1.25, 1.28 and 1.05 ms; 3.40,
// 3.15, 4.97, 4.58 and 3.76 ms: two or four rows of a thread lie too far apart
// to share lines of the L1, and bands of 64 rows are cut up less well.
// Batches: two rows, wavefronts of 16 x 4 (bands of 32 rows): 16 problems of
// 96 rows and 6 of 240, whole SIRT calls, 7.68 and 26.6 ms against 8.02 and
// 27.3 with 1 x 32 and 8.43 and 31.1 with 2 x 64.
struct FpLanes {
  int32_t rpt, row_shift;
};
FpLanes fp_lanes(int32_t rows, int32_t rpt, bool batch) {
  if (rpt != 1 && rpt != 2 && rpt != 4) rpt = batch && rows > 16 ? 2 : 1;
  int32_t s = batch || rpt == 4 ? 4 : 5;
  while (s > 0 && (1 << (s - 1)) >= rows) --s;  // few rows: more columns
  return {rpt, s};
}

// Validate one forward-projection problem and fill its kernel arguments
// for `lanes` and workgroup groups of at most `cap_angles` x
// `cap_cols` column tiles.
int make_fp_args(const kk::FpSpec& S, FpLanes lanes, int32_t cols_per_block,
                 int32_t cap_angles, int32_t cap_cols, FpArgs& A) {
  using kk::fail;
  if (S.plan == nullptr || !S.plan->fp_set)
    return fail(KK_ERR_NOT_SET,
                "Please set the projection geometry with `set_params()`.");
  if (S.tex == nullptr || (S.out == nullptr && S.ptrs == nullptr))
    return fail(KK_ERR_INVALID, "kk_cone_fp: null argument");
  if (S.ptrs != nullptr &&
      (S.mode == 2 || S.out_dual != 0 || S.ptr_axis < 0 || S.ptr_axis > 2))
    return fail(KK_ERR_INVALID,
                "kk_cone_fp_ptrs: a pointer table takes plain or additive "
                "output along axis 0, 1 or 2");
  if (S.rows <= 0 || S.cols <= 0)
    return fail(KK_ERR_INVALID, "kk_cone_fp: bad detector size");
  if (S.mode == 2 && (S.y == nullptr || S.R == nullptr))
    return fail(KK_ERR_INVALID, "kk_cone_fp: residual mode needs y and R");
  if (S.mode == 1 && S.out_dual != 0)
    return fail(KK_ERR_INVALID, "kk_cone_fp: dual output is write-only");
  A = FpArgs{};
  A.tex = reinterpret_cast<const char*>(S.tex);
  A.out = S.out;
  A.out_ptrs = S.ptrs;
  A.ptr_axis = S.ptr_axis;
  A.os0 = S.ptrs != nullptr && S.ptr_axis == 0 ? 0 : S.os[0];
  A.os1 = S.ptrs != nullptr && S.ptr_axis == 1 ? 0 : S.os[1];
  A.os2 = S.ptrs != nullptr && S.ptr_axis == 2 ? 0 : S.os[2];
  A.out_dual = S.out_dual;
  if (S.mode == 2) {
    A.y = S.y;
    A.ys0 = S.ys[0];
    A.ys1 = S.ys[1];
    A.ys2 = S.ys[2];
    A.R = S.R;
    A.rs0 = S.rs[0];
    A.rs1 = S.rs[1];
    A.rs2 = S.rs[2];
  }
  A.rows = S.rows;
  A.cols = S.cols;
  A.n_angles = S.plan->fp_n;
  A.row_shift = lanes.row_shift;
  const int32_t band = lanes.rpt << lanes.row_shift;
  const int32_t wide = cols_per_block << (6 - lanes.row_shift);
  A.row_tiles = (S.rows + band - 1) / band;
  A.col_tiles = (S.cols + wide - 1) / wide;
  A.mode = S.mode;
  A.grp_a = group_size(A.n_angles, cap_angles);
  A.grp_c = group_size(A.col_tiles, cap_cols);
  A.xcd_group = A.grp_a * A.grp_c;
  A.total_blocks = int64_t(A.row_tiles) *
                   ((A.n_angles + A.grp_a - 1) / A.grp_a) * A.grp_a *
                   ((A.col_tiles + A.grp_c - 1) / A.grp_c) * A.grp_c;
  if (A.total_blocks >= (int64_t(1) << 31))
    return fail(KK_ERR_UNSUPPORTED, "kk_cone_fp: grid too large");
  return KK_OK;
}

// Many problems, one launch: a persistent grid walks the concatenated
// workgroup tiles of all problems; a tile finds its problem by binary
// search over the problems' first tile ids (wave-uniform).
struct FpItem {
  const kk::FpAngle* tab;
  FpArgs args;
};

template <int R, bool ALL_COLC, bool FAR>
__global__ __launch_bounds__(kColsBatch * kWave, fp_waves(R)) void cone_fp_batch_kernel(
    const FpItem* __restrict__ items, const int64_t* __restrict__ first,
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
    const FpItem& it = items[lo];
    const int64_t local = g - first[lo];
    fp_tile<R, ALL_COLC, fp_pipe(R), kColsBatch, true, FAR>(it.tab, it.args,
               kk_xcd_remap(local, it.args.total_blocks, it.args.xcd_group));
  }
}

// Whether the plan has an axis of more than kSegment slices.
bool fp_far(const kk_plan_s* plan) {
  for (int a = 0; a < 3; ++a)
    if ((plan->fp_mask & (1 << a)) && plan->fp_shape[a] > kSegment)
      return true;
  return false;
}

}  // namespace

namespace kk {

struct FpBatch {
  FpItem* items = nullptr;
  int64_t* first = nullptr;
  int32_t n = 0;
  int64_t total = 0;
  int32_t rpt = 4;
  bool all_colc = false;
  bool far = false;
};

int fp_batch_build(const std::vector<FpSpec>& specs, int32_t rows_per_thread,
                   FpBatch** out) {
  if (specs.empty()) return fail(KK_ERR_INVALID, "empty forward batch");
  int32_t max_rows = 0;
  for (const FpSpec& S : specs) max_rows = S.rows > max_rows ? S.rows : max_rows;
  bool far = false;
  for (const FpSpec& S : specs)
    far = far || (S.plan != nullptr && S.plan->fp_set && fp_far(S.plan));
  const FpLanes lanes = fp_lanes(max_rows, far ? 1 : rows_per_thread, true);
  std::vector<FpItem> items(specs.size());
  std::vector<int64_t> first(specs.size());
  int64_t total = 0;
  for (size_t p = 0; p < specs.size(); ++p) {
    const int rc = make_fp_args(specs[p], lanes, kColsBatch, kGroupAngles,
                                kGroupColsBatch, items[p].args);
    if (rc != KK_OK) return rc;
    items[p].tab = specs[p].plan->fp;
    first[p] = total;
    total += items[p].args.total_blocks;
  }
  auto* b = new (std::nothrow) FpBatch();
  if (b == nullptr) return fail(KK_ERR_INVALID, "out of host memory");
  b->n = static_cast<int32_t>(specs.size());
  b->total = total;
  b->rpt = lanes.rpt;
  b->far = far;
  b->all_colc = true;
  for (const FpSpec& S : specs) b->all_colc = b->all_colc && S.plan->fp_all_colc;
  hipError_t e = hipMalloc(&b->items, sizeof(FpItem) * items.size());
  if (e == hipSuccess) e = hipMalloc(&b->first, sizeof(int64_t) * first.size());
  if (e == hipSuccess)
    e = hipMemcpy(b->items, items.data(), sizeof(FpItem) * items.size(),
                  hipMemcpyHostToDevice);
  if (e == hipSuccess)
    e = hipMemcpy(b->first, first.data(), sizeof(int64_t) * first.size(),
                  hipMemcpyHostToDevice);
  if (e != hipSuccess) {
    fp_batch_free(b);
    return hip_fail(e, "forward batch descriptors");
  }
  *out = b;
  return KK_OK;
}

void fp_batch_free(FpBatch* b) {
  if (b == nullptr) return;
  if (b->items) hipFree(b->items);
  if (b->first) hipFree(b->first);
  delete b;
}

int fp_batch_launch(const FpBatch* b, int32_t grid_blocks,
                    hipStream_t stream) {
  if (b == nullptr) return fail(KK_ERR_NOT_SET, "forward batch not built");
  int64_t g = grid_blocks > 0 ? grid_blocks : b->total;
  if (g > b->total) g = b->total;
  if (g <= 0) return KK_OK;
  const dim3 grid(static_cast<unsigned>(g));
  auto* kernel =
      b->far        ? &cone_fp_batch_kernel<1, false, true>
      : b->rpt == 1 ? &cone_fp_batch_kernel<1, false, false>
      : b->rpt == 2 ? (b->all_colc ? &cone_fp_batch_kernel<2, true, false>
                                   : &cone_fp_batch_kernel<2, false, false>)
                    : (b->all_colc ? &cone_fp_batch_kernel<4, true, false>
                                   : &cone_fp_batch_kernel<4, false, false>);
  hipLaunchKernelGGL(kernel, grid, dim3(kColsBatch * kWave), 0, stream,
                     b->items, b->first, b->n, b->total);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return hip_fail(e, "cone_fp_batch_kernel");
  return KK_OK;
}

}  // namespace kk

namespace kk {

int fp_spec(FpSpec& S, const kk_plan* plan, const float* tex, float* out,
            const int64_t os[3], int32_t rows, int32_t cols,
            int32_t additive) {
  if (os == nullptr) return fail(KK_ERR_INVALID, "kk_cone_fp: null strides");
  S = FpSpec{};
  S.plan = plan;
  S.tex = tex;
  S.out = out;
  for (int t = 0; t < 3; ++t) S.os[t] = os[t];
  S.rows = rows;
  S.cols = cols;
  S.mode = additive ? 1 : 0;
  return KK_OK;
}

int sirt_residual_spec(FpSpec& S, const kk_plan* plan, const float* x_tex,
                       const float* y, const int64_t ys[3], const float* R,
                       const int64_t rs[3], float* res_tex, int32_t n_angles,
                       int32_t rows, int32_t cols) {
  if (plan == nullptr || !plan->fp_set)
    return fail(KK_ERR_NOT_SET, "kk_sirt_fp_residual: no parameters");
  if (n_angles != plan->fp_n)
    return fail(KK_ERR_SHAPE, "kk_sirt_fp_residual: angle count");
  if (res_tex == nullptr || ys == nullptr || rs == nullptr)
    return fail(KK_ERR_INVALID, "kk_sirt_fp_residual: null argument");
  // write the residual straight into the backprojection texture: P(a, r, c)
  // is component 0 of element (a, r+1, c+1) and component 1 of (a, r, c+1)
  const int64_t tc = cols + kHalo, tr = rows + kHalo;
  S = FpSpec{};
  S.plan = plan;
  S.tex = x_tex;
  S.out = res_tex + 2 * (kHaloLo * tc + kHaloLo);
  S.os[0] = 2 * tr * tc;
  S.os[1] = 2 * tc;
  S.os[2] = 2;
  S.out_dual = 1 - 2 * tc;
  S.rows = rows;
  S.cols = cols;
  S.mode = 2;
  S.y = y;
  S.R = R;
  for (int t = 0; t < 3; ++t) {
    S.ys[t] = ys[t];
    S.rs[t] = rs[t];
  }
  return KK_OK;
}

}  // namespace kk

namespace {

int launch_fp_spec(const kk::FpSpec& S, hipStream_t stream) {
  FpArgs A;
  const int rc = make_fp_args(S, fp_lanes(S.rows, 0, false), kColsSingle,
                              kGroupAngles, kGroupCols, A);
  if (rc != KK_OK) return rc;
  const dim3 grid(static_cast<unsigned>(A.total_blocks));
  const dim3 block(kColsSingle * kWave);
  const bool far = fp_far(S.plan), ptrs = S.ptrs != nullptr;
  auto* kernel = far ? (ptrs ? &cone_fp_kernel<true, true>
                             : &cone_fp_kernel<true, false>)
                     : (ptrs ? &cone_fp_kernel<false, true>
                             : &cone_fp_kernel<false, false>);
  hipLaunchKernelGGL(kernel, grid, block, 0, stream, S.plan->fp, A);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return kk::hip_fail(e, "cone_fp_kernel");
  return KK_OK;
}

// Rows per thread of the line kernel for `rows` detector rows at the plan's
// c spacing (0: the launch is the gather kernel's).  Costs in cycles of a
// SIMD, fitted on MI355X over 1400 circular geometries (volumes of 24 to 512
// voxels, 1 to 400 angles, spacings of 0.4 to 2 voxels; calls with their texture
// builds): a slice costs the line kernel's wavefront 72 + 30 R, the gather 66
// per 64 rows, and more where its lanes spread over the cache lines (spacing
// above 1), less so if the volume's pairs stay in the caches (one frame up to
// kGatherCached bytes).
// * The gather's wavefronts are 32 rows (fewer for fewer rows) by two columns
//   or more, the line kernel's 64 rows of one: 388 slices, 308 angles, 4 rows
//   at a spacing of 1.3 voxels 0.19 ms by gathers and 1.31 by lines, 32 rows at
//   512^2 x 32, 360 angles 1.21 and 3.29.  Beyond 32 rows of a volume that the
//   caches don't hold, both come in steps of 64 rows.
// * Launches of few workgroups are as long as one wavefront: a slice takes 0.2
//   us by gathers, 0.35 by lines.  256^3, one angle of 384^2 98 and 135 us, three
//   angles 233 and 176; 128^3, 16 angles of 160^2 56 and 77 us, 64 angles 118 and
//   110.  (Where pairs have to be built of a large volume the line is lower:
//   they are twice the bytes.  Volumes of a few slices are as long as the call's
//   host part either way.)
// * kGatherCached: 197 x 244 x 197, 82 rows, 158 angles (75 MB of pairs) 381 us by
//   lines and 458 by gathers.
constexpr int64_t kGatherCached = 64 << 20;
constexpr int64_t kGatherFew = 600, kGatherFewCached = 2500;  // workgroups
constexpr int32_t kGatherSlices = 64;
int line_rows_per_thread(const kk_plan_s* plan, int32_t rows, int32_t cols) {
  if (!plan->fp_set || plan->fp_line_max < 0.0 || cols > plan->fp_line_cols ||
      rows > plan->fp_line_rows)
    return 0;
  int64_t frame = 0;   // bytes of the largest frame of pairs
  int32_t slices = 0;  // and of slices
  for (int a = 0; a < 3; ++a) {
    if (!(plan->fp_mask & (1 << a))) continue;
    frame = std::max(frame, 8 * kk::frame_elems(plan->fp_shape, a));
    slices = std::max(slices, plan->fp_shape[a]);
  }
  const FpLanes g = fp_lanes(rows, 0, false);
  const int32_t g_rows = g.rpt << g.row_shift;
  const int32_t g_cols = kColsSingle << (6 - g.row_shift);
  const int32_t g_tiles = (rows + g_rows - 1) / g_rows;
  const bool cached = slices >= kGatherSlices && frame <= kGatherCached;
  if (slices >= kGatherSlices &&
      int64_t(plan->fp_n) * g_tiles * ((cols + g_cols - 1) / g_cols) <=
          (cached ? kGatherFewCached : kGatherFew))
    return 0;
  const int32_t groups = (rows + kWave - 1) / kWave;
  const double spread = (cached ? 0.6 : 1.9) *
                        std::max(0.0, plan->fp_line_mean - 1.0);
  int best = 0;
  double best_cost =
      66.2 * (1.0 + spread) *
      (cached || rows <= 32 ? g_tiles * g_rows / double(kWave) : groups);
  for (int r = 1; r <= 4; ++r) {
    // the widest window must fit (its ends' rounding and margins: 4)
    const int32_t span = std::min(kWave * r, rows) - 1;
    if (span * plan->fp_line_max + 4.0 > kLineWords) break;
    const double cost = (72.0 + 30.0 * r) * ((groups + r - 1) / r);
    if (cost < best_cost) {
      best = r;
      best_cost = cost;
    }
  }
  return best;
}

template <bool P>
void launch_line(int32_t r, dim3 grid, hipStream_t stream,
                 const kk::FpAngle* tab, const FpArgs& A) {
  const dim3 block(kLineWaves * kWave);
  switch (r) {
    case 1:
      hipLaunchKernelGGL((cone_fp_line_kernel<1, P>), grid, block, 0, stream,
                         tab, A);
      break;
    case 2:
      hipLaunchKernelGGL((cone_fp_line_kernel<2, P>), grid, block, 0, stream,
                         tab, A);
      break;
    case 3:
      hipLaunchKernelGGL((cone_fp_line_kernel<3, P>), grid, block, 0, stream,
                         tab, A);
      break;
    default:
      hipLaunchKernelGGL((cone_fp_line_kernel<4, P>), grid, block, 0, stream,
                         tab, A);
      break;
  }
}

int launch_fp_planes(const kk::FpSpec& S, hipStream_t stream) {
  if (S.plan == nullptr || !S.plan->fp_set)
    return kk::fail(KK_ERR_NOT_SET,
                    "Please set the projection geometry with `set_params()`.");
  const int32_t r = line_rows_per_thread(S.plan, S.rows, S.cols);
  if (r == 0)
    return kk::fail(KK_ERR_UNSUPPORTED,
                    "kk_cone_fp_planes: not a geometry for planes (see "
                    "kk_fp_reads_planes)");
  FpArgs A;
  const int rc = make_fp_args(S, {r, 6}, kLineWaves, kLineGroupAngles,
                              kLineGroupCols, A);
  if (rc != KK_OK) return rc;
  const dim3 grid(static_cast<unsigned>(A.total_blocks));
  if (S.ptrs != nullptr)
    launch_line<true>(r, grid, stream, S.plan->fp, A);
  else
    launch_line<false>(r, grid, stream, S.plan->fp, A);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return kk::hip_fail(e, "cone_fp_line_kernel");
  return KK_OK;
}

}  // namespace

extern "C" int32_t kk_fp_reads_planes(const kk_plan* plan, int32_t rows,
                                      int32_t cols) {
  if (plan == nullptr || rows <= 0 || cols <= 0) return 0;
  return line_rows_per_thread(plan, rows, cols) > 0 ? 1 : 0;
}

extern "C" int kk_cone_fp_planes(const kk_plan* plan, const float* planes,
                                 float* proj, const int64_t* ptrs,
                                 int32_t ptr_axis, const int64_t ps[3],
                                 int32_t rows, int32_t cols, int32_t additive,
                                 void* stream) {
  kk::FpSpec S;
  const int rc = kk::fp_spec(S, plan, planes, proj, ps, rows, cols, additive);
  if (rc != KK_OK) return rc;
  S.ptrs = ptrs;
  S.ptr_axis = ptr_axis;
  return launch_fp_planes(S, static_cast<hipStream_t>(stream));
}

extern "C" int kk_cone_fp(const kk_plan* plan, const float* vol_tex,
                          float* proj, const int64_t ps[3], int32_t rows,
                          int32_t cols, int32_t additive, void* stream) {
  kk::FpSpec S;
  const int rc = kk::fp_spec(S, plan, vol_tex, proj, ps, rows, cols,
                             additive);
  if (rc != KK_OK) return rc;
  return launch_fp_spec(S, static_cast<hipStream_t>(stream));
}

extern "C" int kk_cone_fp_ptrs(const kk_plan* plan, const float* vol_tex,
                               const int64_t* ptrs, int32_t ptr_axis,
                               const int64_t ps[3], int32_t rows,
                               int32_t cols, int32_t additive, void* stream) {
  if (ptrs == nullptr)
    return kk::fail(KK_ERR_INVALID, "kk_cone_fp_ptrs: null pointer table");
  kk::FpSpec S;
  const int rc = kk::fp_spec(S, plan, vol_tex, nullptr, ps, rows, cols,
                             additive);
  if (rc != KK_OK) return rc;
  S.ptrs = ptrs;
  S.ptr_axis = ptr_axis;
  return launch_fp_spec(S, static_cast<hipStream_t>(stream));
}

extern "C" int kk_sirt_fp_residual(const kk_plan* plan, const float* x_tex,
                                   const float* y, const int64_t ys[3],
                                   const float* R, const int64_t rs[3],
                                   float* res_tex, int32_t n_angles,
                                   int32_t rows, int32_t cols, void* stream) {
  kk::FpSpec S;
  const int rc = kk::sirt_residual_spec(S, plan, x_tex, y, ys, R, rs,
                                        res_tex, n_angles, rows, cols);
  if (rc != KK_OK) return rc;
  return launch_fp_spec(S, static_cast<hipStream_t>(stream));
}
