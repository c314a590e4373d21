// Device-side geometry, cell lookup and affine products for the CPA kernels.
//
// Rounding contract: every floating-point operation here is a single IEEE
// double operation in the order the reference writes it (no FMA
// contraction; the translation unit is built with -ffp-contract=off and the
// pragma below), so a lookup on the GPU returns the same cell as the
// reference's compute_cell_idx for every input (cpab/gpu/calc_2Dto2D.cu:38-153,
// calc_1Dto1D.cu:62-65, calc_3Dto3D.cu:43-137).
//
// Two forms of each lookup:
//   * LIT  : any increment.  The reference's fmod and divisions, decided from
//            the exact quotient and remainder by an fma (quot_rem), with the
//            divisions themselves only where a decision is within rounding.
//   * POW2 : used when every increment is a power of two.  Then x / inc and
//            x * (1/inc) are the same real number, hence round identically,
//            and fmod(x, inc) / inc == s - trunc(s) with s = x * (1/inc)
//            exactly, while (x - fmod(x, inc)) / inc == trunc(s) exactly
//            (|s| < 2^53; the clamps keep it so or make the difference
//            irrelevant).  The POW2 form therefore returns bit-identical cell
//            ids at a fraction of the cost: no divisions, no fmod loop.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#pragma clang fp contract(off)

namespace cpab {

constexpr int TESS_I = 1;   // triangles / tetrahedra (reference TESS_TYPE 1)
constexpr int TESS_II = 2;  // intervals / rectangles / boxes (TESS_TYPE 2)

// Everything the lookups need, precomputed on the host the way the
// reference kernels compute it inline.
struct Geom {
  int nC0, nC1, nC2, pad;
  double inc_x, inc_y, inc_z;
  double rinc_x, rinc_y, rinc_z;  // 1 / inc: exact for powers of two, else rounded
  double top_x, top_y, top_z;     // clamps nC0*inc_x-1e-10, nC1*inc_y-1e-10, nC2*inc_x-1e-10
  double wall_x, wall_y;          // nC0*inc_x, nC1*inc_y (2D type I out-of-domain tests)
  double eps;                     // margin of CellBounds, in increments
  double sc1, sc17;               // 1 / (1 - 2 eps), 1 / (17 - eps): its scales (2D type I)
  double rn0, rn01;               // 1 / nC0, 1 / (nC0 nC1) (box_of)
};

__device__ __forceinline__ double dmin(double a, double b) { return __builtin_fmin(a, b); }

// Product of two non-negative ints below 2^24 (cell and box indices are far
// below that): the masks let the compiler use v_mul_u32_u24 (full rate)
// instead of v_mul_lo_u32.
__device__ __forceinline__ int mul24(int a, int b) {
  return (int)(((unsigned)a & 0xffffffu) * ((unsigned)b & 0xffffffu));
}
__device__ __forceinline__ double dmax(double a, double b) { return __builtin_fmax(a, b); }

// The exact quotient and remainder of x >= 0 by inc: returns k = floor(x / inc)
// and r = x - k inc = fmod(x, inc), without a division.  k0 = trunc(x * rinc)
// (rinc the rounded reciprocal) is k or off by one: x * rinc is within 2^-52
// relative of x / inc, and k counts only below 2^24 (a larger one is clamped
// by the caller).  x - k0 inc is then r, r - inc or r + inc; the fma gives the
// first two exactly (multiples of the smaller ulp, no larger than inc) and
// rounds the last, if at all, without crossing inc, so its sign against 0 and
// inc tells the case and the remainder is formed again with the right k.
// The lookup is bound by VALU issue, and an IEEE FP64 division is about a
// dozen instructions: with fmod, the index and the in-box coordinate each
// dividing (three per axis), calc_T on MI355X took 277 us for 640 x 480
// points (2D type I), 470 us for 10^6 points (1D, 50 cells) and 562 us for
// 491 520 points (3D type I, with the remap); this way 175, 274 and 331 us.
__device__ __forceinline__ double quot_rem(double x, double inc, double rinc, double& r) {
  double k = __builtin_trunc(x * rinc);
  r = __builtin_fma(-k, inc, x);
  if ((r < 0.0) | (r >= inc)) {  // rare: x within rounding of a multiple of inc
    k = r < 0.0 ? k - 1.0 : k + 1.0;
    r = __builtin_fma(-k, inc, x);
  }
  return k;
}

// One axis of the type II / 1D lookup:
//   round(min(nC-1, max(0, (p - fmod(p, inc)) / inc)))
// p - fmod(p, inc) is trunc(p / inc) multiples of inc, and its rounded
// quotient by inc is within 1/2 of that count, so the result is the count
// clamped to [0, nC-1]; fmod of +-inf or NaN is NaN, which max(0, NaN) turns
// into 0.
template <bool POW2>
__device__ __forceinline__ int axis_box(double p, int nC, double inc, double rinc) {
  if (POW2) {
    const double q = __builtin_isfinite(p) ? __builtin_trunc(p * rinc) : 0.0;
    return (int)__builtin_round(dmin((double)(nC - 1), dmax(0.0, q)));
  }
  // k0 = trunc(q * rinc) is off by one at most next to a multiple of inc
  // (quot_rem); a count past nC - 1 stays there whatever its remainder reads
  const double q = dmax(0.0, p);
  const double k0 = __builtin_trunc(q * rinc);
  const double r = __builtin_fma(-k0, inc, q);
  int k = (int)dmin((double)nC, k0);
  k += r >= inc ? 1 : (r < 0.0 ? -1 : 0);
  k = k > nC - 1 ? nC - 1 : k;
  return __builtin_isfinite(p) ? k : 0;
}

// One clamped axis of the type I lookups: the box index (mymin of
// (p0 - xmod) / inc, calc_2Dto2D.cu:20-22) and the in-box coordinate: frac =
// xmod / inc (POW2), or the remainder xmod itself, whose division the caller
// puts off (triangle_of, cell3).
template <bool POW2>
__device__ __forceinline__ int axis_simplex(double p0, int nC, double inc, double rinc, double& frac) {
  int i;
  if (POW2) {
    // p0 >= 0 (clamped), so s >= 0: s - trunc(s) is exact and equals
    // fract(s) = s - floor(s) (one v_fract_f64), and (int)s truncates.
    const double s = p0 * rinc;
    frac = __builtin_amdgcn_fract(s);
    i = (int)s;
  } else {
    i = (int)quot_rem(p0, inc, rinc, frac);
  }
  return i < nC - 1 ? i : nC - 1;
}

template <bool POW2>
__device__ __forceinline__ double divinc(double v, double inc, double rinc) {
  return POW2 ? v * rinc : v / inc;
}

// ------------------------------------------------------------------ 1D
// calc_1Dto1D.cu:62-65
template <bool POW2>
__device__ __forceinline__ int cell1(const double* p, const Geom& g) {
  return axis_box<POW2>(p[0], g.nC0, g.inc_x, g.rinc_x);
}

// ------------------------------------------------------------------ 2D
// Triangle of the point with in-box coordinates x, y (0 top, 1 right, 2
// bottom, 3 left): the reference's tests x < y and 1 - x < y.  Without POW2
// x and y come as the exact remainders and the reference's are their rounded
// quotients by inc.  The products with rinc are within 2^-52 + 2^-54 of
// those, so where both differences exceed 2^-50 they decide the same; only
// next to a diagonal are the quotients formed.
template <bool POW2>
__device__ __forceinline__ int triangle_of(double x, double y, const Geom& g) {
  if (!POW2) {
    const double xa = x * g.rinc_x, ya = y * g.rinc_y;
    const double d1 = xa - ya, d2 = (1.0 - xa) - ya;
    if (__builtin_fabs(d1) > 0x1p-50 & __builtin_fabs(d2) > 0x1p-50)
      return (d1 < 0.0) ? ((d2 < 0.0) ? 2 : 3) : ((d2 < 0.0) ? 1 : 0);
    x = x / g.inc_x;
    y = y / g.inc_y;
  }
  const double omx = 1.0 - x;
  if (x < y) return (omx < y) ? 2 : 3;
  return (omx < y) ? 1 : 0;
}

// calc_2Dto2D.cu:38-153
// FAST (POW2 type I only): when every lane of the wave is strictly inside
// (0, top) on both axes, min(top, max(0, p)) is p, trunc(p / inc) <= nC - 1
// and no outside rule applies, so the lookup is done without the clamps,
// the index mins and the min/max operand canonicalisations IEEE mode needs.
// The test is wave-uniform: a wave with a lane on or past the boundary (or
// NaN) runs the general lookup only.  Measured on MI355X: 256 registration
// chains +14-17 %, one chain with deep speculation +1-2 %, calc_T's redo
// phase +0-3 %; but one chain one step per launch -15 %, so a registration
// launch chooses it.
template <int TESS, bool POW2, bool FAST = false, bool EARLY = true>
__device__ __forceinline__ int cell2(const double* p, const Geom& g) {
  if (TESS == TESS_II) {
    return axis_box<POW2>(p[0], g.nC0, g.inc_x, g.rinc_x) +
           mul24(axis_box<POW2>(p[1], g.nC1, g.inc_y, g.rinc_y), g.nC0);
  }
  const double px = p[0], py = p[1];
  if (POW2 && FAST) {
    // The interior form's cell.  EARLY: formed before the test that allows
    // it, so that the test's scalar chain and branch are off the cell's
    // critical path (a lane outside gets a value that is not used; measured
    // on MI355X: one registration chain +1.2 %, but 256 registration chains
    // one step per launch 2 % slower, so those launches form it after the
    // test).
    const uint64_t ex = __builtin_amdgcn_read_exec();
    if (EARLY) {
      const double sx = px * g.rinc_x, sy = py * g.rinc_y;  // > 0 inside: fract as in axis_simplex
      const double x = __builtin_amdgcn_fract(sx), y = __builtin_amdgcn_fract(sy);
      const int c = ((int)sx + mul24((int)sy, g.nC0)) * 4;
      const double omx = 1.0 - x;
      const int cf = c + ((x < y) ? ((omx < y) ? 2 : 3) : ((omx < y) ? 1 : 0));
      // the strict-interior test as lane masks (fcmp predicates: 2 ordered
      // greater, 4 ordered less; inactive lanes read 0), combined in scalar code
      const uint64_t ok = __builtin_amdgcn_fcmp(px, 0.0, 2) & __builtin_amdgcn_fcmp(px, g.top_x, 4) &
                          __builtin_amdgcn_fcmp(py, 0.0, 2) & __builtin_amdgcn_fcmp(py, g.top_y, 4);
      if ((ok & ex) == ex) return cf;
    } else {
      const uint64_t ok = __builtin_amdgcn_fcmp(px, 0.0, 2) & __builtin_amdgcn_fcmp(px, g.top_x, 4) &
                          __builtin_amdgcn_fcmp(py, 0.0, 2) & __builtin_amdgcn_fcmp(py, g.top_y, 4);
      if ((ok & ex) == ex) {
        const double sx = px * g.rinc_x, sy = py * g.rinc_y;
        const double x = __builtin_amdgcn_fract(sx), y = __builtin_amdgcn_fract(sy);
        const int c = ((int)sx + mul24((int)sy, g.nC0)) * 4;
        const double omx = 1.0 - x;
        if (x < y) return c + ((omx < y) ? 2 : 3);
        return c + ((omx < y) ? 1 : 0);
      }
    }
  }
  const double p0 = dmin(g.top_x, dmax(0.0, px));
  const double p1 = dmin(g.top_y, dmax(0.0, py));
  double x, y;
  const int i = axis_simplex<POW2>(p0, g.nC0, g.inc_x, g.rinc_x, x);
  const int j = axis_simplex<POW2>(p1, g.nC1, g.inc_y, g.rinc_y, y);
  int c = (i + mul24(j, g.nC0)) * 4;  // triangles: 0 top, 1 right, 2 bottom, 3 left
  const bool left = px <= 0.0, right = px >= g.wall_x, up = py <= 0.0, down = py >= g.wall_y;
  if (left | right | up | down) {  // rare: outside the domain
    // the reference's rules, as selects on the four sides' tests
    bool upL = false, dnL = false, upR = false, dnR = false;
    if (POW2 || ((left | right) & (up | down))) {  // (without POW2 four divisions: past a corner only)
      const double nC0 = (double)g.nC0, nC1 = (double)g.nC1;
      const double sx = divinc<POW2>(px, g.inc_x, g.rinc_x), sy = divinc<POW2>(py, g.inc_y, g.rinc_y);
      const double nx = divinc<POW2>(-px, g.inc_x, g.rinc_x), ny = divinc<POW2>(-py, g.inc_y, g.rinc_y);
      upL = up & (sy < sx);
      dnL = down & (sy - nC1 > nx);
      upR = up & (ny > sx - nC0);
      dnR = down & (sy - nC1 > sx - nC0);
    }
    const int tl = upL ? 0 : (dnL ? 2 : 3);
    const int tr = upR ? 0 : (dnR ? 2 : 1);
    const int tm = up ? 0 : 2;
    return c + (left ? tl : (right ? tr : tm));
  }
  return c + triangle_of<POW2>(x, y, g);
}

// cell2's general type I path without branches: the inside and outside
// classifications are both computed and one is selected, so a lane that is
// alone in its wave (a single dependent chain, see lone_trips) pays no
// branch and no strict-interior test.  Same result as cell2 for every point.
// Power-of-two increments only (the others' divisions are better left out).
__device__ __forceinline__ int cell2_flat(const double* p, const Geom& g) {
  constexpr bool POW2 = true;
  const double px = p[0], py = p[1];
  const double p0 = dmin(g.top_x, dmax(0.0, px));
  const double p1 = dmin(g.top_y, dmax(0.0, py));
  double x, y;
  const int i = axis_simplex<POW2>(p0, g.nC0, g.inc_x, g.rinc_x, x);
  const int j = axis_simplex<POW2>(p1, g.nC1, g.inc_y, g.rinc_y, y);
  const int c = (i + mul24(j, g.nC0)) * 4;
  const bool left = px <= 0.0, right = px >= g.wall_x, up = py <= 0.0, down = py >= g.wall_y;
  const double nC0 = (double)g.nC0, nC1 = (double)g.nC1;
  const double sx = divinc<POW2>(px, g.inc_x, g.rinc_x), sy = divinc<POW2>(py, g.inc_y, g.rinc_y);
  const double nx = divinc<POW2>(-px, g.inc_x, g.rinc_x), ny = divinc<POW2>(-py, g.inc_y, g.rinc_y);
  const bool upL = up & (sy < sx), dnL = down & (sy - nC1 > nx);
  const bool upR = up & (ny > sx - nC0), dnR = down & (sy - nC1 > sx - nC0);
  const int tl = upL ? 0 : (dnL ? 2 : 3);
  const int tr = upR ? 0 : (dnR ? 2 : 1);
  const int tm = up ? 0 : 2;
  const int tout = left ? tl : (right ? tr : tm);
  const double omx = 1.0 - x;
  const int tin = (x < y) ? ((omx < y) ? 2 : 3) : ((omx < y) ? 1 : 0);
  return c + ((left | right | up | down) ? tout : tin);
}

// ------------------------------------------------------------------ 3D
// calc_3Dto3D.cu:43-137
template <int TESS, bool POW2>
__device__ __forceinline__ int cell3(const double* p, const Geom& g) {
  if (TESS == TESS_II) {
    const int a = axis_box<POW2>(p[0], g.nC0, g.inc_x, g.rinc_x);
    const int b = axis_box<POW2>(p[1], g.nC1, g.inc_y, g.rinc_y);
    const int cc = axis_box<POW2>(p[2], g.nC2, g.inc_z, g.rinc_z);
    return a + mul24(b, g.nC0) + mul24(cc, mul24(g.nC1, g.nC0));
  }
  const double p0 = dmin(g.top_x, dmax(0.0, p[0]));
  const double p1 = dmin(g.top_y, dmax(0.0, p[1]));
  const double p2 = dmin(g.top_z, dmax(0.0, p[2]));  // top_z uses inc_x, as the reference
  double x, y, z;
  const int i = axis_simplex<POW2>(p0, g.nC0, g.inc_x, g.rinc_x, x);
  const int j = axis_simplex<POW2>(p1, g.nC1, g.inc_y, g.rinc_y, y);
  const int k = axis_simplex<POW2>(p2, g.nC2, g.inc_z, g.rinc_z, z);
  int c = mul24(i + mul24(j, g.nC0) + mul24(k, mul24(g.nC1, g.nC0)), 5);
  // alternating orientation: flip when the parity of i + j + k is odd
  const bool tf = ((i + j + k) & 1) != 0;
  if (!POW2) {
    // the remainders' products with rinc decide unless one of the four planes
    // is within their error (three coordinates of 2^-52 + 2^-54 and the sums'
    // roundings, below 2^-48), as in triangle_of
    const double xa = x * g.rinc_x, ya = y * g.rinc_y, za = z * g.rinc_z;
    const double u = tf ? ya : xa, v = tf ? 1.0 - xa : ya;
    const double d1 = za - u - v, d2 = u + v + za - 2.0, d3 = v - u - za, d4 = u - v - za;
    if (__builtin_fabs(d1) > 0x1p-48 & __builtin_fabs(d2) > 0x1p-48 & __builtin_fabs(d3) > 0x1p-48 &
        __builtin_fabs(d4) > 0x1p-48)
      return c + (d1 > 0.0 ? 1 : (d2 > 0.0 ? 2 : (d3 > 0.0 ? 3 : (d4 > 0.0 ? 4 : 0))));
    x = x / g.inc_x;
    y = y / g.inc_y;
    z = z / g.inc_z;
  }
  if (tf) {
    const double tmp = x;
    x = y;
    y = 1.0 - tmp;
  }
  if (-x - y + z >= 0.0) return c + 1;
  if (x + y + z - 2.0 >= 0.0) return c + 2;
  if (-x + y - z >= 0.0) return c + 3;
  if (x - y - z >= 0.0) return c + 4;
  return c;
}

template <int DIM, int TESS, bool POW2, bool FAST = false, bool EARLY = true>
__device__ __forceinline__ int cell_of(const double* p, const Geom& g) {
  if (DIM == 1) return cell1<POW2>(p, g);
  if (DIM == 2) return cell2<TESS, POW2, FAST, EARLY>(p, g);
  return cell3<TESS, POW2>(p, g);
}

// The box with index b: its place along each axis, as doubles.  b + 1/2 is at
// least half a count from a multiple of n, so the products' rounding (b < 2^24)
// never changes the floors.
template <int DIM>
__device__ __forceinline__ void box_of(int b, const Geom& g, double* k) {
  double r = (double)b;
  if (DIM == 3) {
    const double n01 = (double)mul24(g.nC0, g.nC1);
    k[2] = __builtin_floor((r + 0.5) * g.rn01);
    r = __builtin_fma(-n01, k[2], r);
  }
  if (DIM >= 2) {
    k[1] = __builtin_floor((r + 0.5) * g.rn0);
    r = __builtin_fma(-(double)g.nC0, k[1], r);
  }
  k[0] = r;
}

// ------------------------------------------------------ affine products
// calc_2Dto2D.cu:24-36, calc_1Dto1D.cu:18-52, calc_3Dto3D.cu:25-39
template <int DIM>
__device__ __forceinline__ void affine(double* x, const double* A, const double* b) {
  if (DIM == 1) {
    x[0] = A[0] * b[0] + A[1];
  } else if (DIM == 2) {
    x[0] = A[0] * b[0] + A[1] * b[1] + A[2];
    x[1] = A[3] * b[0] + A[4] * b[1] + A[5];
  } else {
    x[0] = A[0] * b[0] + A[1] * b[1] + A[2] * b[2] + A[3];
    x[1] = A[4] * b[0] + A[5] * b[1] + A[6] * b[2] + A[7];
    x[2] = A[8] * b[0] + A[9] * b[1] + A[10] * b[2] + A[11];
  }
}

template <int DIM>
__device__ __forceinline__ void linear(double* x, const double* A, const double* b) {
  if (DIM == 1) {
    x[0] = A[0] * b[0];
  } else if (DIM == 2) {
    x[0] = A[0] * b[0] + A[1] * b[1];
    x[1] = A[3] * b[0] + A[4] * b[1];
  } else {
    x[0] = A[0] * b[0] + A[1] * b[1] + A[2] * b[2];
    x[1] = A[4] * b[0] + A[5] * b[1] + A[6] * b[2];
    x[2] = A[8] * b[0] + A[9] * b[1] + A[10] * b[2];
  }
}

}  // namespace cpab
