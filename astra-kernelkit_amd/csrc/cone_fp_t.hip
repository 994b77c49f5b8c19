// Exact transpose of the ray-driven (Joseph) forward projection: the
// matched adjoint A^T of kk_cone_fp, for gradients.
//
// The reference has no such operator: its autograd backward uses the
// voxel-driven backprojector (kernelkit/torch_support.py:29-33), which is
// not the transpose of the forward projector.  Here every voxel sums, over
// the (ray, slice) samples of the forward kernel that touch it, the ray's
// value times the ray weight times the sample's bilinear weight for that
// voxel.  Rays and ray weights are the forward kernel's (kk_fp_ray,
// kk_fp_weight); sample coordinates are float32 offsets from float64 anchors at
// the lane's voxels, where the forward kernels step in 64-bit fixed point.  A
// sample's weight so agrees to ~1e-6, and <A x, y> = <x, A^T y> up to that.
//
// MI355X design, two launches per ray axis group:
// 1. ray_weight_kernel: y * (ray weight), 0 for rays the forward kernel
//    skips, written column-major ([angle][col][row]) into the caller's
//    workspace through an LDS tile.  The gather below then reads, for one
//    column, the rows of 64 neighbouring voxels: a few cache lines per
//    wavefront instead of 64.
// 2. A gather, so that no atomics are needed (an LDS float atomic add costs
//    ~190 cycles per wavefront instruction on this part, against ~8 for a
//    plain LDS read-modify-write).  A lane owns 8 voxels along b by 2
//    consecutive ones along c of one slice, summed over all angles of the
//    launch's ray axis and written once.  Owning two c voxels, a lane
//    evaluates each of its samples once for both (a sample has two c taps):
//    3/2 evaluations per sample instead of 2.
//    * cone_fp_t_col_kernel, circular orbits ("column-coherent" angles: the
//      row step has no a/b part): below.
//    * cone_fp_t_kernel, other geometries: each lane projects the support
//      rectangle of its voxels (at its slice) onto the detector and walks
//      the pixels of the bounding box, a column's rows unrolled; the b taps,
//      whose index differs per lane, are summed in the lane's own LDS words
//      (one read-modify-write of three taps per column instead of a select
//      over all registers).
//    A plan with both kinds of angles launches both; each skips the other's.
// Candidate intervals are widened by 1e-6 voxel in coordinate space, far
// above the float64 rounding of the sample coordinates; samples outside
// the support get zero weight.
#include <algorithm>
#include <type_traits>

#include "kk_internal.h"

namespace {

constexpr int kJB = 8;       // voxels along b per lane
constexpr int kJC = 2;       // consecutive voxels along c per lane
constexpr double kEps = 1e-6;

struct FptArgs {
  const float* yw;        // weighted projections [angle][col][row]
  float* vol;
  int64_t sa, sb, sc;     // volume strides along the frame axes a, b, c
  int32_t rows, cols;
  int32_t na, nb, nc;
  int32_t tiles_b, tiles_c;
  const int32_t* angles;  // angle ids of this ray axis
  int32_t n_angles;
  int32_t mode;           // 0: vol = A^T y, 1: vol += A^T y
};

// Angles per cone_fp_t_kernel launch.  A workgroup walks every angle of
// its launch, so the resident workgroups (which start and retire at
// different times) are spread over all of them; neighbouring slices read
// nearly the same pixels of an angle, but share them in the caches only
// if few angles are in flight.  A launch takes the angles whose workspace
// fits this budget (three quarters of MI355X's 256 MiB last-level cache;
// each launch after the first adds to the volume, one read-modify-write
// of it per launch).
constexpr int64_t kChunkBytes = int64_t(192) << 20;
// Consecutive slices of one tile per XCD run (measured on MI355X at
// 1024^3 / 1440 wobbling angles: 4.41 s with 32, 4.38-4.56 s with 16 and
// 64, 5.24 s with 128, 5.44 s with workgroups dealt round-robin in
// c-tile-fastest order).
constexpr int32_t kSliceRun = 32;

constexpr int kTile = 64;  // ray_weight_kernel: 64 x 64 pixels per block
// Zero rows before and after every column of the workspace: a lane's row
// window of up to kRowPad rows may start above or end below the detector
// and still reads in-bounds zeros, so the column loop needs no per-row
// bounds test.
constexpr int kRowPad = 16;

// yw[angle][col][kRowPad + row] = proj(angle, row, col) * kk_fp_weight of
// the ray, 0 where kk_fp_ray rejects the ray, and kRowPad zeros before and
// after each column (column stride rows + 2 kRowPad).  Reads along columns
// and writes along rows, both coalesced, through an LDS tile.
__global__ __launch_bounds__(256) void ray_weight_kernel(
    const kk::FpAngle* __restrict__ tab, const float* __restrict__ proj,
    int64_t ps0, int64_t ps1, int64_t ps2, int32_t rows, int32_t cols,
    int32_t tiles_r, int32_t tiles_c, float* __restrict__ yw) {
  __shared__ float tile[kTile][kTile + 1];
  int64_t bid = blockIdx.x;
  const int32_t tcol = static_cast<int32_t>(bid % tiles_c);
  bid /= tiles_c;
  const int32_t trow = static_cast<int32_t>(bid % tiles_r);
  const int32_t ang = static_cast<int32_t>(bid / tiles_r);
  const kk::FpAngle& P = tab[ang];
  const int32_t lane = threadIdx.x & 63;
  const int32_t w = threadIdx.x >> 6;
  const int32_t r0 = trow * kTile, c0 = tcol * kTile;
  const float* img = proj + ang * ps0;
  for (int32_t t = w; t < kTile; t += 4) {
    const int32_t r = r0 + t, col = c0 + lane;
    float v = 0.f;
    if (r < rows && col < cols) {
      double a1, b1, a2, b2;
      if (kk_fp_ray(P, r, col, a1, b1, a2, b2))
        v = img[r * ps1 + col * ps2] * kk_fp_weight(P, a1, a2);
    }
    tile[t][lane] = v;
  }
  __syncthreads();
  const int64_t cs = rows + 2 * kRowPad;
  float* out = yw + static_cast<int64_t>(ang) * cols * cs + kRowPad;
  for (int32_t t = w; t < kTile; t += 4) {
    const int32_t col = c0 + t, r = r0 + lane;
    if (col >= cols) continue;
    if (r < rows) out[col * cs + r] = tile[lane][t];
    // the pads: above the first row band, below the last
    if (trow == 0 && lane < kRowPad) out[col * cs - kRowPad + lane] = 0.f;
    if (trow == tiles_r - 1 && lane < kRowPad)
      out[col * cs + rows + lane] = 0.f;
  }
}

// 1 / d in float64 for the detector boxes and the walk's anchor: the
// hardware estimate and one Newton step, which squares its relative error
// (to ~1e-14 from the estimate's ~1e-7: far below the 1e-6 voxel widening
// of the boxes and the float32 rounding of the anchor offsets); non-finite
// for d = 0.
__device__ __forceinline__ double rcp64(double d) {
  const double r = __builtin_amdgcn_rcp(d);
  return fma(r, fma(-d, r, 1.0), r);
}

// 1 / d to the last bits: a second Newton step.
__device__ __forceinline__ double rcp64x2(double d) {
  const double r = rcp64(d);
  return fma(r, fma(-d, r, 1.0), r);
}

// Least / greatest value over a wavefront whose 64 lanes are all active
// (DPP steps and a readlane, no LDS round trips), as a scalar.
__device__ __forceinline__ int32_t wave_min_all(int32_t v) {
  return __builtin_amdgcn_readfirstlane(__reduce_min_sync(~0ull, v));
}
__device__ __forceinline__ int32_t wave_max_all(int32_t v) {
  return __builtin_amdgcn_readfirstlane(__reduce_max_sync(~0ull, v));
}

// Integer interval [ceil(lo), floor(hi)] clipped to [0, n - 1].
__device__ __forceinline__ void int_range(double lo, double hi, int32_t n,
                                          int32_t& a, int32_t& b) {
  lo = fmax(lo, -1.0);
  hi = fmin(hi, static_cast<double>(n));
  a = max(0, static_cast<int32_t>(ceil(lo)));
  b = min(n - 1, static_cast<int32_t>(floor(hi)));
}
__device__ __forceinline__ void int_range(float lo, float hi, int32_t n,
                                          int32_t& a, int32_t& b) {
  lo = fmaxf(lo, -1.f);
  hi = fminf(hi, static_cast<float>(n));
  a = max(0, static_cast<int32_t>(ceilf(lo)));
  b = min(n - 1, static_cast<int32_t>(floorf(hi)));
}

// Ends a run of samples whose b tap index is the float t: S - T goes to
// tap row t and T to row t + 1 of the lane's b-tap sums, then the run is
// cleared.  g has a spare row on either side (rows -1 and kJB, never
// written out), so the four read-modify-writes need no bounds branches
// and are issued together (two paired LDS reads, two paired writes, one
// round trip).  A run whose index is outside [-1, kJB) (outside the b-run,
// the "no run yet" marker -2, non-finite coordinates) adds zeros to rows
// -1 and 0.
__device__ __forceinline__ void close_run(float (*g)[kJC][64], int32_t lane,
                                          float t, float* S, float* T) {
  static_assert(kJC == 2, "close_run covers two c voxels per lane");
  const bool in = t >= -1.f && t < static_cast<float>(kJB);
  const int32_t row = in ? static_cast<int32_t>(t) : -1;
  float* p = &g[row][0][lane];
  const float a0 = in ? S[0] - T[0] : 0.f, a1 = in ? S[1] - T[1] : 0.f;
  const float b0 = in ? T[0] : 0.f, b1 = in ? T[1] : 0.f;
  // rows are kJC * 64 words apart, c voxels 64 words
  const float v0 = p[0], v1 = p[64], v2 = p[128], v3 = p[192];
  p[0] = v0 + a0;
  p[64] = v1 + a1;
  p[128] = v2 + b0;
  p[192] = v3 + b1;
#pragma unroll
  for (int cc = 0; cc < kJC; ++cc) S[cc] = T[cc] = 0.f;
}

// Consecutive rows of a column, at any element alignment.
typedef float f32x2_u __attribute__((ext_vector_type(2), aligned(4)));
typedef float f32x3_u __attribute__((ext_vector_type(3), aligned(4)));
typedef float f32x4_u __attribute__((ext_vector_type(4), aligned(4)));

// max(0, 1 - |x|), one instruction (|x| and the clamp to [0, 1] are free)
__device__ __forceinline__ float tent(float x) {
  float w;
  asm("v_sub_f32_e64 %0, 1.0, |%1| clamp" : "=v"(w) : "v"(x));
  return w;
}

// min(max(x, 0), 1), 0 for NaN, one instruction
__device__ __forceinline__ float unit(float x) {
  float w;
  asm("v_max_f32_e64 %0, %1, %1 clamp" : "=v"(w) : "v"(x));
  return w;
}
__device__ __forceinline__ float unit_neg(float x) {
  float w;
  asm("v_max_f32_e64 %0, -%1, -%1 clamp" : "=v"(w) : "v"(x));
  return w;
}

// W consecutive rows, four per load
template <int W>
__device__ __forceinline__ void load_rows(const char* p, float* y) {
#pragma unroll
  for (int t = 0; t < W; t += 4) {
    if (t + 4 <= W) {
      const f32x4_u v = *reinterpret_cast<const f32x4_u*>(p + 4 * t);
#pragma unroll
      for (int e = 0; e < 4; ++e) y[t + e] = v[e];
    } else if (t + 3 == W) {
      const f32x3_u v = *reinterpret_cast<const f32x3_u*>(p + 4 * t);
      y[t] = v[0];
      y[t + 1] = v[1];
      y[t + 2] = v[2];
    } else if (t + 2 == W) {
      const f32x2_u v = *reinterpret_cast<const f32x2_u*>(p + 4 * t);
      y[t] = v[0];
      y[t + 1] = v[1];
    } else {
      y[t] = *reinterpret_cast<const float*>(p + 4 * t);
    }
  }
}

// Value of lane `l` of a wavefront (l wave-uniform), in scalar registers.
__device__ __forceinline__ int32_t bcast(int32_t v, int32_t l) {
  return __builtin_amdgcn_readlane(v, l);
}

// Other geometries.
//
// Bound by vector instructions: about 20 per row of a column and lane, 55 per
// column (coordinates, three b taps read, added to and written back in LDS),
// and the lanes whose box has fewer rows or columns than the wavefront's
// largest idle for the difference.  So a column's rows are unrolled (four per
// load, no loop or per-row test), the reciprocal of the perspective is taken
// once per column, and the b taps go to LDS once per column; row by row, with
// a reciprocal each and a run of equal b taps flushed wherever one lane's tap
// changed (40 % of the rows), a row took about 37 slots.
// A workgroup is one b-run of one slice whose wavefronts share out the angles:
// enough wavefronts for small volumes, and shorter float32 sums.
// Measured (one launch per axis, wobbling angles, before -> now): 256^3 / 360
// angles of 384^2 19.4 -> 12.7 ms, 128^3 / 128 of 192^2 1.59 -> 0.67 ms,
// 64^3 / 64 of 96^2 0.75 -> 0.13 ms; of that the unrolled columns 13.7 -> 10.0
// and the shares 10.0 -> 9.1 ms at 256^3 / 256 angles.
//
// Workgroups from which the angles go to 4 shares, and to 8 (fewer: 16).
// Measured in ms for 4 / 8 / 16 shares: 128 workgroups 0.095 / 0.067 / 0.053,
// 512 0.178 / 0.133 / 0.129, 1152 0.40 / 0.34 / 0.37, 2048 0.77 / 0.67 / 0.80,
// 3400 1.52 / 1.50 / 1.81, 8280 3.17 / 3.21 / 4.36, 16384 9.1 / 9.1 / 12.0.
// No more shares than hold the angles: wavefronts without any cost the others
// their places.  In us with 1 / 2 / 4 / 8 / 16 shares, angles of a launch: 8192
// workgroups, one angle 64 / 78 / 114 / 209 / 533, 2 angles 197 / 198 / 260 / 449
// / 1152, 4 angles 323 / 324 / 335 / 463 / 1197; 2048, 2 angles 58 / 48 / 59 / 76
// / 161, 4 angles 84 / 66 / 66 / 80 / 169; 512, 2 angles 51 / 41 / 40 / 40 / 52, 8
// angles 127 / 86 / 61 / 49 / 59 (all but the first: calls of two launches).
constexpr int64_t kGenShares4 = 4096, kGenShares8 = 640;

template <int SHARES>
__global__ __launch_bounds__(64 * SHARES, 6) void cone_fp_t_kernel(
    const kk::FpAngle* __restrict__ tab, FptArgs A) {
  // slice fastest, then b tile, then c tile; runs of kSliceRun
  // consecutive ids (neighbouring slices of one tile, which read nearly
  // the same pixels of every angle) go to one XCD, so its L2 serves them
  const int64_t total = int64_t(A.na) * A.tiles_b * A.tiles_c;
  int64_t bid = kk_xcd_remap(blockIdx.x, total, kSliceRun);
  const int32_t i = static_cast<int32_t>(bid % A.na);
  bid /= A.na;
  const int32_t tb = static_cast<int32_t>(bid % A.tiles_b);
  const int32_t tc = static_cast<int32_t>(bid / A.tiles_b);
  const int32_t lane = threadIdx.x & 63;
  const int32_t k = (tc * 64 + lane) * kJC;  // first of the lane's c voxels
  const int32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int32_t jw = tb * kJB;
  const int32_t per = (A.n_angles + SHARES - 1) / SHARES;
  const int32_t q_end = min(A.n_angles, (wave + 1) * per);

  const double fi = static_cast<double>(i);
  const double kd = static_cast<double>(k);
  const int32_t cstride = A.rows + 2 * kRowPad;  // workspace column stride
  const int64_t angle_elems = static_cast<int64_t>(cstride) * A.cols;
  // b-tap sums of this lane's voxels (row t: b voxel jw + t), indexed per
  // lane: every lane owns its words, so no atomics and no cross-lane
  // ordering are needed; taps just outside the b-run are not written out.
  // The run flushes use a spare row on either side of it (g[-1], g[kJB]).
  constexpr int kSpare = 1;
  __shared__ float gacc[SHARES][kJB + 2 * kSpare][kJC][64];
  float(*g)[kJC][64] = gacc[wave] + kSpare;
#pragma unroll
  for (int t = -kSpare; t < kJB + kSpare; ++t)
#pragma unroll
    for (int cc = 0; cc < kJC; ++cc) g[t][cc][lane] = 0.f;

  for (int32_t q = wave * per; q < q_end; ++q) {
    const int32_t ang = A.angles[q];
    const kk::FpAngle& P = tab[ang];
    const float* img = A.yw + ang * angle_elems + kRowPad;
    const double arel = fi + P.sig;  // slice centre, relative to the source
    if (P.colc) continue;  // cone_fp_t_col_kernel's
    // pixels whose rays meet the support rectangle of this lane's voxels
    // at this slice: bounding box of its projected corners.  The ray
    // through the source-relative point X meets the detector at
    // col = (V x Q).X / N.X, row = (Q x U).X / N.X with N = U x V
    // (q + col U + row V = lam X, lam = U.(V x Q) / N.X > 0 in front of
    // the source): linear forms in X, whose a and b parts (the slice and
    // the wave's b-run) are shared by the wave; each lane adds its c part.
    const double nva = P.ub * P.vc - P.uc * P.vb;
    const double nvb = P.uc * P.va - P.ua * P.vc;
    const double nvc = P.ua * P.vb - P.ub * P.va;
    const double mva = P.vb * P.qc - P.vc * P.qb;
    const double mvb = P.vc * P.qa - P.va * P.qc;
    const double mvc = P.va * P.qb - P.vb * P.qa;
    const double rva = P.qb * P.uc - P.qc * P.ub;
    const double rvb = P.qc * P.ua - P.qa * P.uc;
    const double rvc = P.qa * P.ub - P.qb * P.ua;
    const double lamn = P.ua * mva + P.ub * mvb + P.uc * mvc;
    double cmin = 1e300, cmax = -1e300, rmin = 1e300, rmax = -1e300;
    bool ok = true;
#pragma unroll
    for (int eb = 0; eb < 2; ++eb) {
      const double xb = (eb ? jw + kJB + 1 + kEps : jw - kEps) - P.taub;
      const double dn = fma(nvb, xb, nva * arel);
      const double cn = fma(mvb, xb, mva * arel);
      const double rn = fma(rvb, xb, rva * arel);
#pragma unroll
      for (int ec = 0; ec < 2; ++ec) {
        const double xc =
            (ec ? kd + (kJC + 1) + kEps : kd - kEps) - P.tauc;
        const double inv = rcp64(fma(nvc, xc, dn));
        const double pc = fma(mvc, xc, cn) * inv;
        const double pr = fma(rvc, xc, rn) * inv;
        ok = ok && isfinite(pc) && isfinite(pr) && lamn * inv > 0.0;
        cmin = fmin(cmin, pc);
        cmax = fmax(cmax, pc);
        rmin = fmin(rmin, pr);
        rmax = fmax(rmax, pr);
      }
    }
    int32_t c_lo = 0, c_hi = A.cols - 1, r_lo = 0, r_hi = A.rows - 1;
    if (ok) {
      int_range(cmin, cmax, A.cols, c_lo, c_hi);
      int_range(rmin, rmax, A.rows, r_lo, r_hi);
    }
    // columns in a loop of wave-uniform length, each lane walking its
    // own column range from its first column (a tilted rotation axis
    // shifts the lanes' ranges against each other: a loop over their
    // union would leave a lane idle for the difference), rows per lane.
    // Sample coordinates: float64 at an anchor pixel
    // (the wave's first column, the lane's first row), float32 offsets
    // from it.  With D = q + col U + row V (kk_fp_ray's terms) and
    // t = D_b / D_a at the anchor, x_b = arel D_b / D_a + tau_b moves by
    // arel (dD_b - t dD_a) / D_a between the anchor and a pixel: a
    // quantity of the box's size, so its float32 rounding is ~1e-6
    // voxel.  Weights are the tents 1 - |x - centre| of the forward
    // kernel's bilinear taps.
    const int32_t wc_lo = wave_min_all(c_lo <= c_hi ? c_lo : A.cols);
    const double fwc = static_cast<double>(wc_lo);
    const double fr0 = static_cast<double>(r_lo);
    const double Da0 = fma(fr0, P.va, fma(fwc, P.ua, P.qa));
    const double Db0 = fma(fr0, P.vb, fma(fwc, P.ub, P.qb));
    const double Dc0 = fma(fr0, P.vc, fma(fwc, P.uc, P.qc));
    const double inv0 = rcp64(Da0);
    const double tb = Db0 * inv0, tcv = Dc0 * inv0;
    const float ob =
        static_cast<float>(fma(tb, arel, P.taub) - (jw + kk::kHaloLo));
    const float oc =
        static_cast<float>(fma(tcv, arel, P.tauc) - (kd + kk::kHaloLo));
    const float da0 = static_cast<float>(Da0);
    const float tbf = static_cast<float>(tb), tcf = static_cast<float>(tcv);
    const float arf = static_cast<float>(arel);
    const float uaf = static_cast<float>(P.ua), ubf = static_cast<float>(P.ub),
                ucf = static_cast<float>(P.uc);
    const float vaf = static_cast<float>(P.va), vbf = static_cast<float>(P.vb),
                vcf = static_cast<float>(P.vc);
    const bool anchor_ok = ok && isfinite(tb) && isfinite(tcv);
    // With u the row offset from the lane's first row and dc the column
    // offset from the wave's first column, dA = dc ua + u va (b, c
    // alike) and x_b = ob + arel (dB - tb dA) / (Da0 + dA): per column
    // the numerator arel (dB - tb dA) is affine in u with slope
    // arel (vb - tb va), and the denominator with slope va (c alike).
    const float kvb = arf * fmaf(-tbf, vaf, vbf);
    const float kvc = arf * fmaf(-tcf, vaf, vcf);
    const int32_t ncol =
        anchor_ok && c_lo <= c_hi && r_lo <= r_hi ? c_hi - c_lo + 1 : 0;
    const int32_t wncol = wave_max_all(ncol);
    const int32_t wnrow = wave_max_all(ncol > 0 ? r_hi - r_lo + 1 : 0);
    // Short windows, all rows of a column unrolled: with g(u) = u / (1 +
    // eps u) and eps = va / den at the column's first row, both
    // coordinates are A + B g.  eps u is tiny for any usual geometry, so g
    // takes three terms of its series (what is left out, B u (eps u)^3, is
    // below 1e-7 voxel by the bound here), and the window's samples span
    // less than one voxel along b: three tap rows from the floor of the
    // smaller end, added to the lane's words once per column.
    {
      // (with the rows that fill the window up to an unrolled length)
      const float w = static_cast<float>(
          wnrow <= 8 ? wnrow : (wnrow <= 12 ? 12 : kRowPad));
      const float d1 = fmaf(static_cast<float>(c_lo - wc_lo), uaf, da0);
      const float d2 = fmaf(static_cast<float>(c_hi - wc_lo), uaf, da0);
      const float dm = fminf(fabsf(d1), fabsf(d2));
      // (the slopes B are kvb / den and kvc / den up to the offsets inside
      // the box, which eps makes small)
      const bool fit = wnrow <= kRowPad && d1 * d2 > 0.f &&
                       fabsf(vaf) * w <= 2e-3f * dm &&
                       fabsf(kvb) * w <= 0.9f * dm &&
                       fabsf(kvc) * w <= 16.f * dm;
      if (__ballot(ncol > 0 && !fit) == 0) {
        auto walk = [&](auto ww) {
          constexpr int W = decltype(ww)::value;
          uint32_t o = 4u * (static_cast<uint32_t>(c_lo) *
                                 static_cast<uint32_t>(cstride) +
                             static_cast<uint32_t>(r_lo));
          float dcf = static_cast<float>(c_lo - wc_lo);
          for (int32_t j = 0; j < wncol; ++j) {
            if (j < ncol) {
              asm volatile("" : "+v"(o));
              float y[W];
              load_rows<W>(reinterpret_cast<const char*>(img) + o, y);
              const float dAc = dcf * uaf;
              const float rc = __builtin_amdgcn_rcpf(da0 + dAc);
              const float ab = arf * fmaf(-tbf, dAc, dcf * ubf) * rc;
              const float ac = arf * fmaf(-tcf, dAc, dcf * ucf) * rc;
              const float Bb = fmaf(-ab, vaf, kvb) * rc;
              const float Bc = fmaf(-ac, vaf, kvc) * rc;
              const float eps = vaf * rc;
              const float xb0 = ab + ob, xc0 = ac + oc;
              const float t0 = __builtin_amdgcn_fmed3f(
                  floorf(fminf(xb0, fmaf(Bb, static_cast<float>(W - 1), xb0))),
                  -1.f, static_cast<float>(kJB - 2));
              // relative to the middle tap row; what lies outside the
              // three rows adds to the spare rows, or nothing
              const float hb0 = xb0 - (t0 + 1.f);
              float P[3][kJC];
#pragma unroll
              for (int r = 0; r < 3; ++r)
#pragma unroll
                for (int cc = 0; cc < kJC; ++cc) P[r][cc] = 0.f;
#pragma unroll
              for (int t = 0; t < W; ++t) {
                const float u = static_cast<float>(t);
                const float gu =
                    t == 0 ? 0.f
                           : fmaf(fmaf(eps, u * u * u, -u * u), eps, u);
                const float xc = t == 0 ? xc0 : fmaf(Bc, gu, xc0);
                const float h = t == 0 ? hb0 : fmaf(Bb, gu, hb0);
                const float u0 = y[t] * tent(xc);
                const float u1 = y[t] * tent(xc - 1.f);
                const float g0 = unit_neg(h), g1 = tent(h), g2 = unit(h);
                P[0][0] = fmaf(u0, g0, P[0][0]);
                P[0][1] = fmaf(u1, g0, P[0][1]);
                P[1][0] = fmaf(u0, g1, P[1][0]);
                P[1][1] = fmaf(u1, g1, P[1][1]);
                P[2][0] = fmaf(u0, g2, P[2][0]);
                P[2][1] = fmaf(u1, g2, P[2][1]);
              }
              float* p = &g[static_cast<int32_t>(t0)][0][lane];
              // rows are kJC * 64 words apart, c voxels 64 words; all
              // reads before the writes
              float v[3 * kJC];
#pragma unroll
              for (int r = 0; r < 3 * kJC; ++r) v[r] = p[64 * r];
#pragma unroll
              for (int r = 0; r < 3 * kJC; ++r)
                p[64 * r] = v[r] + P[r / kJC][r % kJC];
            }
            o += 4u * static_cast<uint32_t>(cstride);
            dcf += 1.f;
          }
        };
        if (wnrow <= 2)
          walk(std::integral_constant<int, 2>{});
        else if (wnrow <= 3)
          walk(std::integral_constant<int, 3>{});
        else if (wnrow <= 4)
          walk(std::integral_constant<int, 4>{});
        else if (wnrow <= 5)
          walk(std::integral_constant<int, 5>{});
        else if (wnrow <= 6)
          walk(std::integral_constant<int, 6>{});
        else if (wnrow <= 7)
          walk(std::integral_constant<int, 7>{});
        else if (wnrow <= 8)
          walk(std::integral_constant<int, 8>{});
        else if (wnrow <= 12)
          walk(std::integral_constant<int, 12>{});
        else
          walk(std::integral_constant<int, kRowPad>{});
        continue;
      }
    }
    // Other windows, row by row: b-tap sums over a run of samples with the
    // same tap index, added to the lane's LDS words when the index changes:
    // S = sum of y w_c, T = sum of y w_c fb, so the taps t and t + 1
    // receive S - T and T.  A run stays open from column to column while
    // the index holds (the sums of one index add up whatever the column),
    // so along the walk a run closes about once per b voxel crossed.  The
    // index is kept as a float (the floor of x_b); a run reaches the LDS
    // words only if its index lies in [-1, kJB) and is dropped otherwise.
    // Rows outside the lane's tents add zeros; a non-finite coordinate (a
    // ray parallel to the slices) starts a run of its own that is dropped.
    float tcur = -2.f;  // no run yet
    float S[kJC], T[kJC];
#pragma unroll
    for (int cc = 0; cc < kJC; ++cc) S[cc] = T[cc] = 0.f;
    // the workspace of this angle as bytes (a wave-uniform base) and a
    // 32-bit byte offset per lane: the launcher keeps an angle's
    // workspace below 4 GiB
    const char* imgb = reinterpret_cast<const char*>(img);
    const uint32_t nrow =
        static_cast<uint32_t>(max(0, r_hi - r_lo + 1));
    for (int32_t j = 0; j < wncol; ++j) {
      const int32_t col = c_lo + j;  // this lane's column (in range if
                                     // j < ncol)
      const float dcf = static_cast<float>(col - wc_lo);
      const float dAc = dcf * uaf;
      const float nb0 = arf * fmaf(-tbf, dAc, dcf * ubf);
      const float nc0 = arf * fmaf(-tcf, dAc, dcf * ucf);
      const float den0 = da0 + dAc;
      uint32_t o = 4u * (static_cast<uint32_t>(col) *
                             static_cast<uint32_t>(cstride) +
                         static_cast<uint32_t>(r_lo));
      const uint32_t oend = o + 4u * (j < ncol ? nrow : 0u);
      float drf = 0.f;
      // four rows per load (what it reads past the lane's box is of the
      // column or its pad)
      for (; o < oend; o += 16u) {
        // The empty asm keeps the offset a 32-bit register (an SGPR base
        // plus a VGPR offset), not a 64-bit pointer stepped per row.
        asm volatile("" : "+v"(o));
        float y[4];
        load_rows<4>(imgb + o, y);
#pragma unroll
        for (int t = 0; t < 4; ++t, drf += 1.f) {
          if (t > 0 && o + 4u * t >= oend) break;
          const float yv = y[t];
          const float rc = __builtin_amdgcn_rcpf(fmaf(drf, vaf, den0));
          const float xc = fmaf(fmaf(drf, kvc, nc0), rc, oc);
          const float xb = fmaf(fmaf(drf, kvb, nb0), rc, ob);
          const float fl = floorf(xb);
          if (fl != tcur) {
            close_run(g, lane, tcur, S, T);
            tcur = fl;
          }
          const float yfb = yv * (xb - fl);
          const float w0 = fmaxf(0.f, 1.f - fabsf(xc));
          const float w1 = __builtin_amdgcn_fmed3f(0.f, xc, 2.f - xc);
          S[0] = fmaf(yv, w0, S[0]);
          S[1] = fmaf(yv, w1, S[1]);
          T[0] = fmaf(yfb, w0, T[0]);
          T[1] = fmaf(yfb, w1, T[1]);
        }
      }
    }
    close_run(g, lane, tcur, S, T);
  }

  // the shares' sums, each wavefront some of the b voxels
  __syncthreads();
  constexpr int kPart = (kJB + SHARES - 1) / SHARES;
  if (wave * kPart >= kJB) return;
#pragma unroll
  for (int cc = 0; cc < kJC; ++cc) {
    const int32_t kc = k + cc;
    if (kc >= A.nc) break;
#pragma unroll
    for (int e = 0; e < kPart; ++e) {
      const int32_t t = wave * kPart + e;
      const int32_t j = jw + t;
      if (j >= A.nb) break;
      float v = 0.f;
#pragma unroll
      for (int s = 0; s < SHARES; ++s) v += gacc[s][t + kSpare][cc][lane];
      const int64_t o = i * A.sa + j * A.sb + kc * A.sc;
      if (A.mode == 1)
        A.vol[o] += v;
      else
        A.vol[o] = v;
    }
  }
}

// ---------------------------------------------------------------------------
// Column-coherent angles (circular orbits).
//
// The b coordinate of a sample depends on the detector column alone, and the
// c coordinate is affine in the row.  So the columns that reach a wavefront's
// 8 b voxels are an interval per angle, the same for all lanes; a column's
// sum over the rows that reach a lane's two c voxels enters two neighbouring
// b voxels with the column's weights.  What bounds it is the number of vector
// instructions and of row loads per (wavefront, column), in balance (profiled
// at 256^3, 360 angles of 384^2: 0.27 vector instructions per SIMD and cycle,
// address unit busy in 76 %):
// * rows come in loads of four per lane (unaligned dwordx4): at the lanes'
//   stride of two voxels a single dword costs the same 16 cycles;
// * the b voxels are registers.  The walk over tap rows is unrolled, so each
//   column adds to registers known at compile time, instead of four LDS
//   read-modify-writes per column;
// * a column's float64 data (about 120 instructions) is computed one column
//   per lane for 64 columns at a time, taken across angles (an angle has
//   about 11 per wavefront), and read back as an LDS broadcast and scalars;
// * the number of rows per window is a template parameter, picked for 64
//   columns at a time, and taps that are outside every lane's tent (the
//   first row's second voxel, the last rows' first) are left out;
// * a workgroup's slices are neighbours, which read nearly the same rows;
//   its other wavefronts share out the angles and are added up at the end,
//   which fills the chip for small volumes (and halves the length of the
//   float32 sums: error against float64 1.3e-7 instead of 2.5e-7).
// Measured with 256^3 / 360 angles of 384^2: 5.2 ms, before 10.2 ms (dword
// row loads, an angle's columns at a time, sums in LDS); 128^3 / 128 angles:
// 0.25 ms, before 0.67 ms; 64^3 / 64 angles: 0.09 ms, before 0.31 ms.
// 16 voxels along b halve the work at run borders, but need a third of the
// wavefronts' room: 7.1 ms.  One c voxel per lane: 7.1 ms.

constexpr int kColSlices = 4;  // slices (wavefronts) per workgroup part
constexpr int kColB = 8;       // voxels along b per lane
// Wavefronts of one part from which a workgroup shares its angles out to two
// parts, below to four (measured, two against four: 16384 5.23 / 5.45 ms,
// 9600 1.26 / 1.24 ms, 2048 0.32 / 0.25 ms, 512 0.12 / 0.09 ms).
constexpr int64_t kColSplit2 = 12288;
// Wavefronts of one part that fill half the chip.  From there a part has six
// angles or more, whose columns fill the 64 that are set up at a time (1 / 2 / 4
// parts in us, angles of a launch: 16384 wavefronts, 4 angles 164 / 193 / 252, 16
// angles 501 / 520 / 565; 9216, 2 angles 90 / 100 / 138, 8 angles 192 / 188 / 212,
// 16 angles 347 / 324 / 334; 4800, 2 angles 40 / 48 / 63); below, no more parts
// than hold the angles (2048, 2 angles 46 / 44 / 46, 8 angles 93 / 74 / 67).
constexpr int64_t kColFill = 4096;
constexpr int kColAngles = 6;
// Marks a column whose record has whole voxels apart (whole_s).
constexpr uint64_t kWhole = uint64_t(1) << 63;

// LONG: for plans whose windows are longer than kRowPad rows on the whole, where
// rows are less than kLongSpacing voxels apart (60 angles of 1152^2 pixels of a
// quarter voxel, 128^3: 11.3 -> 3.8 ms); other plans it would cost 1 to 4%.
constexpr double kLongSpacing = 0.3;
template <int SPLIT, bool LONG>
__global__ __launch_bounds__(64 * kColSlices * SPLIT, 8) void
cone_fp_t_col_kernel(
    const kk::FpAngle* __restrict__ tab, FptArgs A) {
  const int32_t groups = (A.na + kColSlices - 1) / kColSlices;
  const int64_t total = int64_t(groups) * A.tiles_b * A.tiles_c;
  int64_t bid = kk_xcd_remap(blockIdx.x, total, kSliceRun / kColSlices);
  const int32_t wave =
      __builtin_amdgcn_readfirstlane(int32_t(threadIdx.x) >> 6);
  const int32_t sub = wave / kColSlices;
  const int32_t i = static_cast<int32_t>(bid % groups) * kColSlices +
                    wave % kColSlices;
  bid /= groups;
  const int32_t jw = static_cast<int32_t>(bid % A.tiles_b) * kColB;
  const int32_t k0 = static_cast<int32_t>(bid / A.tiles_b) * (64 * kJC);
  const int32_t lane = threadIdx.x & 63;
  const uint32_t cstride = A.rows + 2 * kRowPad;
  const uint64_t angle_elems = static_cast<uint64_t>(cstride) * A.cols;
  // this part's angles (none for slices past the volume)
  const int32_t per = (A.n_angles + SPLIT - 1) / SPLIT;
  const int32_t q_end = i < A.na ? min(A.n_angles, (sub + 1) * per) : 0;

  __shared__ float4 rec_s[kColSlices * SPLIT][64][2];
  __shared__ float whole_s[kColSlices * SPLIT][64];
  __shared__ int3 run_s[kColSlices * SPLIT][64];
  float4(*rec)[2] = rec_s[wave];
  float* whole = whole_s[wave];
  int3* run = run_s[wave];

  float acc[kColB][kJC];
#pragma unroll
  for (int t = 0; t < kColB; ++t)
#pragma unroll
    for (int cc = 0; cc < kJC; ++cc) acc[t][cc] = 0.f;

  for (int32_t q0 = sub * per; q0 < q_end; q0 += 64) {
    // the column intervals of the next 64 angles, one angle per lane:
    // columns whose b coordinate at this slice lies in [jw, jw + kColB + 1);
    // a1 = (x_b - taub) / arel, and for these angles
    // a1 = (col ub + qb) / (col ua + qa)
    // (converted where they are used: kept as doubles for the whole walk,
    // these cost the registers of another resident wavefront)
    int32_t ii = i, jj = jw;
    asm volatile("" : "+s"(ii), "+s"(jj));
    int32_t l_ang = 0, l_lo = 0, l_n = 0;
    if (q0 + lane < q_end) {
      l_ang = A.angles[q0 + lane];
      const kk::FpAngle& P = tab[l_ang];
      if (P.colc) {
        // (reciprocals to ~1e-14, far inside the widening by kEps)
        const double ra = rcp64(static_cast<double>(ii) + P.sig);
        const double t1 = (jj - kEps - P.taub) * ra;
        const double t2 = (jj + kColB + 1 + kEps - P.taub) * ra;
        const double d1 = fma(t1, P.ua, -P.ub), d2 = fma(t2, P.ua, -P.ub);
        int32_t c_lo = 0, c_hi = A.cols - 1;
        if (d1 * d2 > 0.0) {
          const double c1 = fma(-t1, P.qa, P.qb) * rcp64(d1);
          const double c2 = fma(-t2, P.qa, P.qb) * rcp64(d2);
          if (isfinite(c1) && isfinite(c2))
            int_range(fmin(c1, c2), fmax(c1, c2), A.cols, c_lo, c_hi);
        }
        l_lo = c_lo;
        l_n = max(0, c_hi - c_lo + 1);
      }
    }
    // the intervals' columns one after the other: an angle's run starts at
    // the sum of the counts before it
    int32_t end = l_n;
#pragma unroll
    for (int s = 1; s < 64; s <<= 1) {
      const int32_t v = __shfl_up(end, s);
      end += lane >= s ? v : 0;
    }
    const int32_t n_all = bcast(end, 63);
    run[lane] = make_int3(end, l_ang, l_lo - (end - l_n));
    for (int32_t g0 = 0; g0 < n_all; g0 += 64) {
      // column g0 + lane of the runs: its rays (kk_fp_ray's terms: the row
      // terms of a and b are exact zeros for these angles) and the c
      // coordinate of its rows at this slice, beta + alpha r (padded
      // coordinates)
      int32_t t0 = -99, nr = 0;
      uint64_t base = 0;
      float iaf = 0.f, o1 = 0.f, ah = 0.f, al = 0.f, x0 = 0.f, fb = 0.f,
            hi = 0.f, xw = 0.f;
      bool neg = false;
      int32_t is = i, nbs = A.nb + 1, ks = k0 + 1;
      asm volatile("" : "+s"(is), "+s"(nbs), "+s"(ks));
      if (g0 + lane < n_all) {
        int32_t q = 0;   // the first run that ends after g0 + lane
#pragma unroll
        for (int s = 32; s > 0; s >>= 1)
          if (run[q + s - 1].x <= g0 + lane) q += s;
        const int3 r = run[q];
        const kk::FpAngle& P = tab[r.y];
        const int32_t col = r.z + g0 + lane;
        const double fi = static_cast<double>(is);
        const double arel = fi + P.sig;
        const double fc = static_cast<double>(col);
        const double inv = rcp64x2(fma(fc, P.ua, P.qa));
        const double a1 = fma(fc, P.ub, P.qb) * inv;
        const double b1 = fma(a1, P.sig, P.taub);
        const double s = inv * arel;
        double alpha = P.vc * s;
        // c offset of row 0 from the tile's first voxel
        double xb = fma(fma(fc, P.uc, P.qc), s, P.tauc) -
                    static_cast<double>(ks);
        if (isfinite(b1) && isfinite(alpha) && isfinite(xb)) {
          uint32_t ib;
          kk_fp_coord(a1, b1, fi, static_cast<double>(nbs), ib, fb);
          t0 = static_cast<int32_t>(ib) - kk::kHaloLo - jw;
          neg = alpha < 0.0;
          if (neg) {  // mirrored: from the tile's last voxel, downwards
            alpha = -alpha;
            xb = (64 * kJC - 1) - xb;
          }
          ah = static_cast<float>(alpha);
          al = static_cast<float>(alpha - static_cast<double>(ah));
          // A lane's window: the rows whose c coordinate lies in the open
          // span (-1, kJC) of its voxels' tents, (kJC + 1) / alpha rows long,
          // i.e. at most floor(len) + 1 integer rows from the ceiling of
          // the first one, moved 1e-3 row earlier (float32 rounding is
          // below 1e-4 row; rows outside get zero weight).  Longer ones
          // than the zero rows around a column allow are walked lane by
          // lane (nr > kRowPad).
          const double ia = ah > 1e-6f ? rcp64(alpha) : 0.0;
          iaf = static_cast<float>(ia);
          const float len = static_cast<float>(kJC + 1) * iaf;
          nr = iaf == 0.f || len + 3.f > static_cast<float>(kRowPad)
                   ? kRowPad + 1
                   : static_cast<int32_t>(floorf(len + 2e-3f)) + 1;
          const double r1 = (-1.0 - xb) * ia;
          const double rb =
              floor(fmin(fmax(r1, -kRowPad), static_cast<double>(A.rows)));
          o1 = static_cast<float>(fmax(r1 - rb, -1e7)) - 1e-3f;
          // Whole voxels of the offset apart where the base is not the first
          // row of lane 0's window but the detector's edge: kept in x0, they
          // would cost its low bits.
          double xr = fma(alpha, rb, xb);
          if (rb != floor(r1)) {
            xw = static_cast<float>(fmin(fmax(floor(xr), -4e6), 4e6));
            xr -= static_cast<double>(xw);
          }
          x0 = static_cast<float>(xr);
          const int32_t rbi = static_cast<int32_t>(rb);
          hi = static_cast<float>(A.rows - rbi);
          base = r.y * angle_elems + static_cast<uint32_t>(col) * cstride +
                 static_cast<uint32_t>(kRowPad + rbi) +
                 (xw != 0.f ? kWhole : 0);
        }
      }
      rec[lane][0] = make_float4(iaf, o1, ah, al);
      rec[lane][1] = make_float4(x0, hi, fb, 1.f - fb);
      whole[lane] = xw;
      for (int sgn = 0; sgn < 2; ++sgn) {
        const bool mine = t0 != -99 && neg == (sgn != 0);
        if (__ballot(mine) == 0) continue;
        const int32_t tt = mine ? t0 : -99;
        const int32_t nn = mine ? nr : 0;
        const float lv = static_cast<float>(kJC * (sgn ? 63 - lane : lane));
        // one column, windows of at most W rows: the lane's sums over it
        auto column = [&](int32_t l, auto w, auto dr, float* cs, float2& f) {
          constexpr int W = decltype(w)::value;
          constexpr bool D = decltype(dr)::value;
          const uint32_t blo =
              static_cast<uint32_t>(bcast(static_cast<int32_t>(base), l));
          const uint32_t bhi = static_cast<uint32_t>(
              bcast(static_cast<int32_t>(base >> 32), l));
          const float* yc =
              A.yw + (((static_cast<uint64_t>(bhi) << 32) | blo) & ~kWhole);
          const float4 ra = rec[l][0], rb = rec[l][1];
          f = make_float2(rb.z, rb.w);
          const float du = __builtin_amdgcn_fmed3f(
              ceilf(fmaf(lv, ra.x, ra.y)), 0.f, rb.y);
          const char* p = reinterpret_cast<const char*>(yc) +
                          (static_cast<uint32_t>(du) << 2);
          float lx = lv;
          if (bhi >> 31) lx -= whole[l];
          const float x = fmaf(ra.w, du, fmaf(ra.z, du, -lx)) + rb.x;
          if constexpr (W == 0) {
            // rows one by one, in the kernel for long windows four at a time,
            // up to the end of the lane's window (rows past it get zero
            // weight; past the detector, read zeros)
            const float end =
                ra.x == 0.f
                    ? rb.y - 1.f
                    : fminf(floorf(fmaf(lv, ra.x, ra.y) + 2e-2f +
                                   static_cast<float>(kJC + 1) * ra.x),
                            rb.y - 1.f);
            cs[0] = 0.f;
            cs[1] = 0.f;
            if constexpr (!LONG) {
              for (float d = du; d <= end; d += 1.f, p += 4) {
                const float xd = fmaf(ra.w, d, fmaf(ra.z, d, -lx)) + rb.x;
                const float y = *reinterpret_cast<const float*>(p);
                cs[0] = fmaf(y, tent(xd), cs[0]);
                cs[1] = fmaf(y, tent(xd - 1.f), cs[1]);
              }
            } else {
              for (float d = du; d <= end; d += 4.f, p += 16) {
                const float xd = fmaf(ra.w, d, fmaf(ra.z, d, -lx)) + rb.x;
                float y[4];
                load_rows<4>(p, y);
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                  const float xt = fmaf(ra.z, static_cast<float>(t), xd);
                  cs[0] = fmaf(y[t], tent(xt), cs[0]);
                  cs[1] = fmaf(y[t], tent(xt - 1.f), cs[1]);
                }
              }
            }
            return;
          } else {
            float y[W];
            load_rows<W>(p, y);
#pragma unroll
            for (int t = 0; t < W; ++t) {
              const float xt =
                  t == 0 ? x : fmaf(ra.z, static_cast<float>(t), x);
              if (!D || t < (2 * W + 2) / 3)
                cs[0] = t == 0 ? y[t] * tent(xt)
                               : fmaf(y[t], tent(xt), cs[0]);
              const float w1 = __builtin_amdgcn_fmed3f(0.f, xt, 2.f - xt);
              if (t == (D ? 1 : 0))
                cs[1] = y[t] * w1;
              else if (t > 0)
                cs[1] = fmaf(y[t], w1, cs[1]);
            }
          }
        };
        auto walk = [&](auto w, auto dr) {
#pragma unroll
          for (int t = -1; t < kColB; ++t) {
            uint64_t mask = __ballot(tt == t);
            while (mask != 0) {
              const int32_t l = __builtin_ctzll(mask);
              mask &= mask - 1;
              float cs[kJC];
              float2 f;
              column(l, w, dr, cs, f);
              auto add = [&](float c0, float c1) {
                if (t >= 0) acc[t][0] = fmaf(f.y, c0, acc[t][0]);
                if (t + 1 < kColB) acc[t + 1][0] = fmaf(f.x, c0, acc[t + 1][0]);
                if (t >= 0) acc[t][1] = fmaf(f.y, c1, acc[t][1]);
                if (t + 1 < kColB) acc[t + 1][1] = fmaf(f.x, c1, acc[t + 1][1]);
              };
              if (sgn == 0)
                add(cs[0], cs[kJC - 1]);
              else
                add(cs[kJC - 1], cs[0]);
            }
          }
        };
        // below one c voxel per row the first row reaches no lane's second
        // voxel, and the last ones (from 2 / alpha on) no lane's first
        const bool D = __ballot(mine && ah > 0.999f) == 0;
        if (__ballot(nn > (D ? kRowPad : 4)) != 0)
          walk(std::integral_constant<int, 0>{}, std::false_type{});
        else if (!D && __ballot(nn > 2) == 0)
          walk(std::integral_constant<int, 2>{}, std::false_type{});
        else if (!D && __ballot(nn > 3) == 0)
          walk(std::integral_constant<int, 3>{}, std::false_type{});
        else if (!D)
          walk(std::integral_constant<int, 4>{}, std::false_type{});
        else if (__ballot(nn > 4) == 0)
          walk(std::integral_constant<int, 4>{}, std::true_type{});
        else if (__ballot(nn > 5) == 0)
          walk(std::integral_constant<int, 5>{}, std::true_type{});
        else if (__ballot(nn > 6) == 0)
          walk(std::integral_constant<int, 6>{}, std::true_type{});
        else if (__ballot(nn > 7) == 0)
          walk(std::integral_constant<int, 7>{}, std::true_type{});
        else if (__ballot(nn > 8) == 0)
          walk(std::integral_constant<int, 8>{}, std::true_type{});
        else if (__ballot(nn > 12) == 0)
          walk(std::integral_constant<int, 12>{}, std::true_type{});
        else
          walk(std::integral_constant<int, kRowPad>{}, std::true_type{});
      }
    }
  }
  if constexpr (SPLIT > 1) {
    __shared__ float part[kColSlices][kColB * kJC][64];
    for (int s = 1; s < SPLIT; ++s) {
      if (sub == s)
#pragma unroll
        for (int t = 0; t < kColB; ++t)
#pragma unroll
          for (int cc = 0; cc < kJC; ++cc)
            part[wave % kColSlices][t * kJC + cc][lane] = acc[t][cc];
      __syncthreads();
      if (sub == 0)
#pragma unroll
        for (int t = 0; t < kColB; ++t)
#pragma unroll
          for (int cc = 0; cc < kJC; ++cc)
            acc[t][cc] += part[wave % kColSlices][t * kJC + cc][lane];
      __syncthreads();
    }
    if (sub != 0) return;
  }
  if (i >= A.na) return;
#pragma unroll
  for (int cc = 0; cc < kJC; ++cc) {
    const int32_t kc = k0 + lane * kJC + cc;
    if (kc >= A.nc) break;
#pragma unroll
    for (int t = 0; t < kColB; ++t) {
      const int32_t j = jw + t;
      if (j >= A.nb) break;
      const int64_t o = i * A.sa + j * A.sb + kc * A.sc;
      A.vol[o] = A.mode == 1 ? A.vol[o] + acc[t][cc] : acc[t][cc];
    }
  }
}

int64_t col_grid(FptArgs& A) {
  A.tiles_b = (A.nb + kColB - 1) / kColB;
  A.tiles_c = (A.nc + 64 * kJC - 1) / (64 * kJC);
  return int64_t((A.na + kColSlices - 1) / kColSlices) * A.tiles_b * A.tiles_c;
}
int64_t general_grid(FptArgs& A) {
  A.tiles_c = (A.nc + 64 * kJC - 1) / (64 * kJC);
  A.tiles_b = (A.nb + kJB - 1) / kJB;
  return int64_t(A.na) * A.tiles_b * A.tiles_c;
}

int column_parts(int64_t blocks, int32_t n_angles) {
  const int64_t waves = blocks * kColSlices;
  const bool fill = waves >= kColFill;
  int parts = waves >= kColSplit2 ? 2 : 4;
  while (parts > 1 &&
         (fill ? n_angles < kColAngles * parts : 2 * n_angles <= parts))
    parts /= 2;
  return parts;
}
void launch_columns(int parts, bool longer, dim3 grid, hipStream_t st,
                    const kk::FpAngle* tab, const FptArgs& A) {
  auto* kernel = parts == 1   ? (longer ? &cone_fp_t_col_kernel<1, true>
                                        : &cone_fp_t_col_kernel<1, false>)
                 : parts == 2 ? (longer ? &cone_fp_t_col_kernel<2, true>
                                        : &cone_fp_t_col_kernel<2, false>)
                              : (longer ? &cone_fp_t_col_kernel<4, true>
                                        : &cone_fp_t_col_kernel<4, false>);
  hipLaunchKernelGGL(kernel, grid, dim3(64 * kColSlices * parts), 0, st, tab,
                     A);
}
int general_shares(int64_t blocks, int32_t n_angles) {
  int shares = blocks >= kGenShares4 ? 4 : blocks >= kGenShares8 ? 8 : 16;
  while (shares / 2 >= n_angles) shares /= 2;
  return shares;
}
void launch_general(int shares, dim3 grid, hipStream_t st,
                    const kk::FpAngle* tab, const FptArgs& A) {
  auto* kernel = shares == 1   ? &cone_fp_t_kernel<1>
                 : shares == 2 ? &cone_fp_t_kernel<2>
                 : shares == 4 ? &cone_fp_t_kernel<4>
                 : shares == 8 ? &cone_fp_t_kernel<8>
                               : &cone_fp_t_kernel<16>;
  hipLaunchKernelGGL(kernel, grid, dim3(64 * shares), 0, st, tab, A);
}

}  // namespace

int64_t kk::fp_transpose_work_floats(const kk_plan_s* plan, int32_t rows,
                                     int32_t cols) {
  if (plan == nullptr || rows <= 0 || cols <= 0) return -1;
  return int64_t(plan->fp_n) * cols * (rows + 2 * kRowPad);
}

int kk::fp_transpose_launch(const kk_plan_s* plan, const float* proj,
                            const int64_t ps[3], int32_t rows, int32_t cols,
                            float* vol, const int32_t vol_shape[3],
                            const int64_t vs[3], int32_t additive, float* work,
                            hipStream_t st) {
  if (plan == nullptr || !plan->fp_set)
    return kk::fail(KK_ERR_NOT_SET,
                    "Please set the projection geometry with `set_params()`.");
  if (proj == nullptr || ps == nullptr || vol == nullptr ||
      vol_shape == nullptr || vs == nullptr || work == nullptr)
    return kk::fail(KK_ERR_INVALID, "kk_cone_fp_transpose: null argument");
  if (rows <= 0 || cols <= 0)
    return kk::fail(KK_ERR_INVALID, "kk_cone_fp_transpose: bad detector");
  if (int64_t(rows) * cols >= (int64_t(1) << 31))
    return kk::fail(KK_ERR_UNSUPPORTED,
                    "kk_cone_fp_transpose: detector of 2^31 pixels or more");
  // the gather addresses one angle's padded workspace with 32-bit byte
  // offsets
  if (int64_t(cols) * (rows + 2 * kRowPad) * 4 >= (int64_t(1) << 32))
    return kk::fail(KK_ERR_UNSUPPORTED,
                    "kk_cone_fp_transpose: detector of 2^30 padded pixels "
                    "or more");
  for (int t = 0; t < 3; ++t)
    if (vol_shape[t] != plan->fp_shape[t])
      return kk::fail(KK_ERR_SHAPE,
                      "kk_cone_fp_transpose: volume shape differs from the "
                      "one the parameters were set for");
  {
    const int32_t tr = (rows + kTile - 1) / kTile;
    const int32_t tcl = (cols + kTile - 1) / kTile;
    const int64_t blocks = int64_t(plan->fp_n) * tr * tcl;
    if (blocks >= (int64_t(1) << 31))
      return kk::fail(KK_ERR_UNSUPPORTED, "kk_cone_fp_transpose: grid");
    hipLaunchKernelGGL(ray_weight_kernel, dim3(unsigned(blocks)), dim3(256),
                       0, st, plan->fp, proj, ps[0], ps[1], ps[2], rows, cols,
                       tr, tcl, work);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return kk::hip_fail(e, "ray_weight_kernel");
  }
  const int64_t angle_bytes = int64_t(cols) * (rows + 2 * kRowPad) * 4;
  const int32_t chunk = static_cast<int32_t>(std::min<int64_t>(
      INT32_MAX, std::max<int64_t>(1, kChunkBytes / angle_bytes)));
  bool first = true;
  for (int a = 0; a < 3; ++a) {
    const int32_t n = plan->fr_start[a + 1] - plan->fr_start[a];
    if (n == 0) continue;
    const int b = kk::kFrameB[a], c = kk::kFrameC[a];
    FptArgs A{};
    A.yw = work;
    A.vol = vol;
    A.sa = vs[a];
    A.sb = vs[b];
    A.sc = vs[c];
    A.rows = rows;
    A.cols = cols;
    A.na = vol_shape[a];
    A.nb = vol_shape[b];
    A.nc = vol_shape[c];
    for (int32_t q0 = 0; q0 < n; q0 += chunk) {
      A.angles = plan->fr_idx + plan->fr_start[a] + q0;
      A.n_angles = std::min(chunk, n - q0);
      for (int colc = 1; colc >= 0; --colc) {
        if (colc ? !plan->fp_any_colc : plan->fp_all_colc) continue;
        A.mode = (first && !additive) ? 0 : 1;
        first = false;
        const int64_t blocks = colc ? col_grid(A) : general_grid(A);
        if (blocks >= (int64_t(1) << 31))
          return kk::fail(KK_ERR_UNSUPPORTED, "kk_cone_fp_transpose: grid");
        const dim3 grid(static_cast<unsigned>(blocks));
        if (colc)
          launch_columns(column_parts(blocks, A.n_angles),
                         plan->fp_line_max >= 0.0 &&
                             plan->fp_line_mean < kLongSpacing,
                         grid, st, plan->fp, A);
        else
          launch_general(general_shares(blocks, A.n_angles), grid, st,
                         plan->fp, A);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return kk::hip_fail(e, "cone_fp_t_kernel");
      }
    }
  }
  return KK_OK;
}

extern "C" int kk_cone_fp_transpose(const kk_plan* plan, const float* proj,
                                    const int64_t ps[3], int32_t rows,
                                    int32_t cols, float* vol,
                                    const int32_t vol_shape[3],
                                    const int64_t vs[3], int32_t additive,
                                    float* work, void* stream) {
  return kk::fp_transpose_launch(plan, proj, ps, rows, cols, vol, vol_shape,
                                 vs, additive, work,
                                 static_cast<hipStream_t>(stream));
}

extern "C" int64_t kk_cone_fp_transpose_work_elems(const kk_plan* plan,
                                                   int32_t rows,
                                                   int32_t cols) {
  return kk::fp_transpose_work_floats(plan, rows, cols);
}
