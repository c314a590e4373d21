// CDNA4 kernels of the CPA integration path.
//
//  * k_prep        sign * As, dt scaling and the per-cell matrix exponential
//                  in one launch (cpab/cpaNd/_CpaCalcs.py:243-313 +
//                  cpab/gpu/expm/expm_affine_by_series_{2D,3D}.py).
//  * k_integrate   calc_T / calc_trajectory (cpab/gpu/calc_2Dto2D.cu:348-408,
//                  499-556).  One lane owns one point at a time; the per-cell
//                  tables live in LDS.  The reference runs every step as
//                  "Trel proposal, and on a cell change nStepsODE RK2
//                  substeps", which in SIMT form idles 63 lanes of a wave
//                  while one lane does its ten substeps.  Here the lanes of
//                  a wave step together while their points stay in their
//                  cells and redo steps together when they have left them
//                  (`advance`), and lanes that finish take the next points
//                  of their block's range.  Per point, the sequence of IEEE
//                  operations is the reference's.
//  * k_simple      calc_T_simple (calc_2Dto2D.cu:412-445).
//  * k_velocity    calc_v (calc_2Dto2D.cu:561-602).
//  * k_cell_idx    calc_cell_idx (calc_2Dto2D.cu:323-344).
//  * k_remap2d / k_remap3d / k_ssd_partial / k_reduce_ll: remap_fwd and the
//                  Gaussian SSD likelihood in FP32 with an FP64 final sum.
#pragma once
#include "cpab_device.h"

#pragma clang fp contract(off)

namespace cpab {

// ------------------------------------------------------------------ expm
// expm_affine_by_series_2D.py:28-74
__device__ inline void expm_2x2(double a, double b, double c, double d, double* E) {
  const double delta_tmp = (a - d) * (a - d) + 4 * b * c;
  const double e = exp((a + d) / 2);
  if (delta_tmp == 0) {
    E[0] = (1 + (a - d) / 2) * e;
    E[1] = b * e;
    E[2] = c * e;
    E[3] = (1 - (a - d) / 2) * e;
  } else if (delta_tmp > 0) {
    const double delta = sqrt(delta_tmp) / 2;
    const double ch = cosh(delta), s = sinh(delta) / delta;
    E[0] = (ch + (a - d) / 2 * s) * e;
    E[1] = b * s * e;
    E[2] = c * s * e;
    E[3] = (ch - (a - d) / 2 * s) * e;
  } else {
    const double delta = sqrt(-delta_tmp) / 2;
    const double co = cos(delta), s = sin(delta) / delta;
    E[0] = (co + (a - d) / 2 * s) * e;
    E[1] = b * s * e;
    E[2] = c * s * e;
    E[3] = (co - (a - d) / 2 * s) * e;
  }
}

// expm_affine_by_series_2D.py:85-237 (closed form when the linear part is
// invertible, else the p-term Taylor series of the 2x3 block)
__device__ inline void expm_affine2(const double* A, double* T, int p) {
  const double A00 = A[0], A01 = A[1], A02 = A[2], A10 = A[3], A11 = A[4], A12 = A[5];
  const double det = A00 * A11 - A01 * A10;
  if (det != 0) {
    double E[4];
    expm_2x2(A00, A01, A10, A11, E);
    T[0] = E[0];
    T[1] = E[1];
    T[3] = E[2];
    T[4] = E[3];
    const double i00 = A11 / det, i11 = A00 / det, i01 = -A01 / det, i10 = -A10 / det;
    const double a = i00 * A02 + i01 * A12;
    const double b = i10 * A02 + i11 * A12;
    T[2] = (T[0] - 1) * a + T[1] * b;
    T[5] = T[3] * a + (T[4] - 1) * b;
    return;
  }
  double S[6] = {1, 0, 0, 0, 1, 0};  // identity, then + A^1 + A^2/2! + ...
  double An[6] = {A00, A01, A02, A10, A11, A12};
  for (int k = 0; k < 6; k++) S[k] += An[k];
  int fact = 1;
  for (int i = 2; i <= p; i++) {
    const double B0 = An[0], B1 = An[1], B2 = An[2], B3 = An[3], B4 = An[4], B5 = An[5];
    fact *= i;
    An[0] = A00 * B0 + A01 * B3;
    An[1] = A00 * B1 + A01 * B4;
    An[2] = A00 * B2 + A01 * B5;
    An[3] = A10 * B0 + A11 * B3;
    An[4] = A10 * B1 + A11 * B4;
    An[5] = A10 * B2 + A11 * B5;
    for (int k = 0; k < 6; k++) S[k] += An[k] / fact;
  }
  for (int k = 0; k < 6; k++) T[k] = S[k];
}

// expm_affine_by_series_3D.py:27-219 (series on the 3x4 block)
__device__ inline void expm_affine3(const double* A, double* T, int p) {
  double S[12] = {1, 0, 0, 0, 0, 1, 0, 0, 0, 0, 1, 0};
  double An[12];
  for (int k = 0; k < 12; k++) An[k] = A[k];
  for (int k = 0; k < 12; k++) S[k] += An[k];
  int fact = 1;
  for (int i = 2; i <= p; i++) {
    double B[12];
    for (int k = 0; k < 12; k++) B[k] = An[k];
    fact *= i;
#pragma unroll
    for (int r = 0; r < 3; r++)
#pragma unroll
      for (int col = 0; col < 4; col++)
        An[r * 4 + col] = A[r * 4 + 0] * B[col] + A[r * 4 + 1] * B[4 + col] + A[r * 4 + 2] * B[8 + col];
    for (int k = 0; k < 12; k++) S[k] += An[k] / fact;
  }
  for (int k = 0; k < 12; k++) T[k] = S[k];
}

// Fused prep of cpab/cpaNd/_CpaCalcs.py:243-313: signedAs = sign*As (the
// reference multiplies by -1 only for the inverse), As_dt = signedAs*dt,
// Trels = expm(As_dt); in 1D the closed form of :285-292.  One lane per
// cell; `inst` strides over independent instances (batched callers).
template <int DIM>
__device__ __forceinline__ void prep_cell(const double* __restrict__ A, int sign, double dt, double* sA,
                                          double* T, int p) {
  constexpr int NE = DIM * (DIM + 1);
  double sAdt[NE];
#pragma unroll
  for (int k = 0; k < NE; k++) {
    double v = A[k];
    if (sign == -1) v *= -1;
    sA[k] = v;
    sAdt[k] = v * dt;
  }
  if (DIM == 1) {
    T[0] = exp(sAdt[0]);
    T[1] = sAdt[1];
    if (sA[0] != 0) T[1] = T[1] * (T[0] - 1) / sAdt[0];
  } else if (DIM == 2) {
    expm_affine2(sAdt, T, p);
  } else {
    expm_affine3(sAdt, T, p);
  }
}

template <int DIM>
__global__ void k_prep(const double* __restrict__ As, int nC, int sign, double dt,
                       double* __restrict__ sA_out, double* __restrict__ T_out, int p,
                       int64_t inst_stride) {
  constexpr int NE = DIM * (DIM + 1);
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= nC) return;
  const int64_t off = (int64_t)blockIdx.y * inst_stride + (int64_t)c * NE;
  double sA[NE], T[NE];
  prep_cell<DIM>(As + off, sign, dt, sA, T, p);
#pragma unroll
  for (int k = 0; k < NE; k++) {
    if (sA_out) sA_out[off + k] = sA[k];
    T_out[off + k] = T[k];
  }
}

// Avees = B theta for m thetas (CpaSpace.theta2Avees, cpab/cpaNd/_CpaSpace.py:366-376):
// one lane per (theta, row), the row's dot product summed in index order, so
// a theta gives the same Avees whatever else is in the batch.  The products'
// operands are loaded eight at a time ahead of the dependent sum (one load
// at a time left the call latency bound: ~30 us for a 3840-row table).
__global__ void k_theta2avees(const double* __restrict__ B, const double* __restrict__ theta,
                              double* __restrict__ Av, int D, int d, int m) {
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (int64_t)m * D) return;
  const int64_t i = idx / D;
  const int r = (int)(idx - i * D);
  const double* row = B + (int64_t)r * d;
  const double* th = theta + i * d;
  double acc = 0.0;
  int j = 0;
  for (; j + 8 <= d; j += 8) {
    double a[8], t[8];
#pragma unroll
    for (int u = 0; u < 8; u++) {
      a[u] = row[j + u];
      t[u] = th[j + u];
    }
#pragma unroll
    for (int u = 0; u < 8; u++) acc += a[u] * t[u];
  }
  for (; j < d; j++) acc += row[j] * th[j];
  Av[idx] = acc;
}

// The reference's gpu_expm(As, Ts, p) on an already scaled table.
template <int DIM>
__global__ void k_expm(const double* __restrict__ As, double* __restrict__ Ts, int nC, int p) {
  constexpr int NE = DIM * (DIM + 1);
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= nC) return;
  double A[NE], T[NE];
#pragma unroll
  for (int k = 0; k < NE; k++) A[k] = As[(int64_t)c * NE + k];
  if (DIM == 2) expm_affine2(A, T, p);
  else expm_affine3(A, T, p);
#pragma unroll
  for (int k = 0; k < NE; k++) Ts[(int64_t)c * NE + k] = T[k];
}

// ------------------------------------------------------------- helpers
__device__ __forceinline__ int lane_id() { return __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0)); }

__device__ __forceinline__ uint64_t ballot(bool b) { return __ballot(b); }

__device__ __forceinline__ int rank_in(uint64_t mask) {
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0));
}

template <int DIM>
__device__ __forceinline__ void load_pt(const double* __restrict__ src, int64_t i, double* p) {
  if (DIM == 2) {
    const double2 v = *reinterpret_cast<const double2*>(src + i * 2);
    p[0] = v.x;
    p[1] = v.y;
  } else {
#pragma unroll
    for (int d = 0; d < DIM; d++) p[d] = src[i * DIM + d];
  }
}

template <int DIM>
__device__ __forceinline__ void store_pt(double* __restrict__ dst, int64_t i, const double* p) {
  if (DIM == 2) {
    *reinterpret_cast<double2*>(dst + i * 2) = make_double2(p[0], p[1]);
  } else {
#pragma unroll
    for (int d = 0; d < DIM; d++) dst[i * DIM + d] = p[d];
  }
}

// Copy the Trel and A tables into LDS (both when they fit).
template <int NE>
__device__ __forceinline__ void stage_tables(double* lds, const double* __restrict__ Trels,
                                             const double* __restrict__ As, int nC) {
  const int n = nC * NE;
  for (int i = threadIdx.x; i < n; i += blockDim.x) {
    lds[i] = Trels ? Trels[i] : 0.0;
    lds[n + i] = As[i];
  }
  __syncthreads();
}

// The per-cell prep fused into a launch (cpab_calc_T_prep): the raw Avees
// table with k_prep's sign and dt.  Every block forms the tables itself
// (prep_cell, the same operations as k_prep) into LDS; block 0 also writes
// them out as cpab_prep_trels would.  raw == nullptr: the tables come ready.
struct PrepSrc {
  const double* raw;
  double* sA_out;
  double* T_out;
  double dt;
  int sign;
};

template <int DIM>
__device__ __forceinline__ void stage_tables_prep(double* lds, const PrepSrc& ps, int nC) {
  constexpr int NE = DIM * (DIM + 1);
  const int n = nC * NE;
  for (int c = threadIdx.x; c < nC; c += blockDim.x) {
    double sA[NE], T[NE];
    prep_cell<DIM>(ps.raw + (int64_t)c * NE, ps.sign, ps.dt, sA, T, 12);
#pragma unroll
    for (int e = 0; e < NE; e++) {
      lds[c * NE + e] = T[e];
      lds[n + c * NE + e] = sA[e];
    }
    if (blockIdx.x == 0) {
#pragma unroll
      for (int e = 0; e < NE; e++) {
        ps.T_out[(int64_t)c * NE + e] = T[e];
        ps.sA_out[(int64_t)c * NE + e] = sA[e];
      }
    }
  }
  __syncthreads();
}

// ---------------------------------------------------------- cell bounds
// Lane masks (bits of inactive lanes are 0); uniform over the wave.
__device__ __forceinline__ uint64_t lanes_lt(double a, double b) { return __builtin_amdgcn_fcmp(a, b, 4); }
__device__ __forceinline__ uint64_t lanes_gt(double a, double b) { return __builtin_amdgcn_fcmp(a, b, 2); }
__device__ __forceinline__ uint64_t lanes_ge(double a, double b) { return __builtin_amdgcn_fcmp(a, b, 3); }
__device__ __forceinline__ uint64_t lanes_lt(int a, int b) { return __builtin_amdgcn_sicmp(a, b, 40); }
__device__ __forceinline__ bool lane_in(uint64_t mask) { return __builtin_amdgcn_inverse_ballot_w64(mask); }

// Whether points are in their cells c, without a lookup: a few affine
// functions of the point against bounds set once for the cell.  The bounds lie
// g.eps inside the cell (the roundings of this test and of the lookup's own
// arithmetic, and the lookup's clamp 1e-10 inside the far walls), so a lane of
// inside(q) is one whose lookup of q gives c; one that is turned down is looked
// up.  NaN and infinite points are turned down.  The box is c's own, from its
// index: one found again from the point can be c's neighbour (a point just
// below a multiple of the increment rounds up in p * (1 / inc)), and a row kept
// within a neighbour's bounds is the wrong one from there on.
//
// Boxes (1D, type II): a lower and an upper bound per axis, none on the sides
// of the domain (the lookup clamps, so what lies beyond belongs to the box).
template <int DIM, int TESS>
struct CellBounds {
  double lo[DIM], hi[DIM];
  __device__ __forceinline__ void enter(int c, const Geom& g) {
    const int nC[3] = {g.nC0, g.nC1, g.nC2};
    const double inc[3] = {g.inc_x, g.inc_y, g.inc_z};
    double k[DIM];
    box_of<DIM>(c, g, k);
#pragma unroll
    for (int d = 0; d < DIM; d++) {
      lo[d] = k[d] > 0.0 ? (k[d] + g.eps) * inc[d] : -__DBL_MAX__;
      hi[d] = k[d] < (double)(nC[d] - 1) ? (k[d] + 1.0 - g.eps) * inc[d] : __DBL_MAX__;
    }
  }
  __device__ __forceinline__ uint64_t inside(const double* q, const Geom&) const {
    uint64_t in = ~0ull;
#pragma unroll
    for (int d = 0; d < DIM; d++) in &= lanes_gt(q[d], lo[d]) & lanes_lt(q[d], hi[d]);
    return in;
  }
};

// 2D triangles, s = p / inc: in triangle k of box (i, j) when u = sx - sy and
// v = sx + sy lie on k's sides of i - j and i + j + 1 (the diagonals) and the
// box edge is not crossed: sy is within the box for top and bottom, sx for
// right and left.  A triangle on the domain's own side instead has the other
// coordinate within the box: the lookup gives everything beyond that side
// above (left of, ...) the box to it, and between the two diagonals the other
// coordinate is within the box anyway.  Past a corner of the domain the
// lookup's border is the diagonal's extension, so there the other coordinate
// is bounded only to keep its rounding small (16 boxes out).
template <>
struct CellBounds<2, TESS_I> {
  double k1, k2, ax, by, mid;
  uint64_t above1, above2;  // lanes whose u lies at or above k1, whose v above k2
  __device__ __forceinline__ void enter(int c, const Geom& g) {
    const double ni = (double)(g.nC0 - 1), nj = (double)(g.nC1 - 1);
    double box[2];
    box_of<2>(c >> 2, g, box);
    const double i = box[0], j = box[1];
    // c & 3: 0 top, 1 right, 2 bottom, 3 left
    const bool b1 = (c & 2) != 0;        // sx - i < sy - j
    const bool b2 = ((c + 1) & 2) != 0;  // their sum > 1
    above1 = ballot(!b1);
    above2 = ballot(b2);
    k1 = (i - j) + (b1 ? -g.eps : g.eps);
    k2 = (i + j + 1.0) + (b2 ? g.eps : -g.eps);
    const bool side = (c & 1) != 0;  // right, left
    const double at = side ? i : j, last = side ? ni : nj;
    const bool onwall = at == (b2 ? last : 0.0);  // (right and bottom look at the far wall)
    const bool usex = side != onwall;
    const double o = usex ? i : j, olast = usex ? ni : nj;
    const bool first = onwall & (o == 0.0), end = onwall & (o == olast);
    const double lo = first ? -16.0 : o + g.eps;
    const double hi = end ? olast + 17.0 : o + 1.0 - g.eps;
    // |w| < 1/2 for lo < s < hi; sc = 1 / (hi - lo)
    const double sc = first & end ? 1.0 / 33.0 : first | end ? g.sc17 : g.sc1;
    ax = usex ? g.rinc_x * sc : 0.0;
    by = usex ? 0.0 : g.rinc_y * sc;
    mid = -0.5 * (lo + hi) * sc;
  }
  __device__ __forceinline__ uint64_t inside(const double* q, const Geom& g) const {
    const double ty = q[1] * g.rinc_y;
    const double u = __builtin_fma(q[0], g.rinc_x, -ty), v = __builtin_fma(q[0], g.rinc_x, ty);
    const double w = __builtin_fma(q[0], ax, __builtin_fma(q[1], by, mid));
    return ~((lanes_ge(u, k1) ^ above1) | (lanes_gt(v, k2) ^ above2)) & lanes_lt(__builtin_fabs(w), 0.5);
  }
};

// 3D tetrahedra: in box (i, j, k) the four corner tetrahedra are cut off by
// the planes sz -+ (sx + sy) and sz +- (sx - sy) at values that depend on the
// box's orientation, and the central one lies on the inner side of all four.
// A corner tetrahedron is bounded by one side of the box per axis besides.
// At the domain's own walls those sides are moved out by half of g.eps (a
// point kept on a wall by zero velocity is within rounding of it, either
// side; the lookup clamps it, which moves each coordinate by at most g.eps,
// hence four of them for the planes) -- but not the far z wall, past which
// the lookup wraps or clamps z at another height (top_z uses inc_x).
template <>
struct CellBounds<3, TESS_I> {
  double k1, k2, k3, k4, fx, fy, fz, zmax;
  uint64_t a1, a2, a3, a4, lx, ly, lz;  // lanes above the planes, lanes whose side is the lower one
  __device__ __forceinline__ void enter(int c, const Geom& g) {
    const double ni = (double)(g.nC0 - 1), nj = (double)(g.nC1 - 1);
    const int b = (int)(((double)c + 0.5) * 0.2), tet = c - mul24(b, 5);  // (a tenth or more from rounding up)
    double box[3];
    box_of<3>(b, g, box);
    const double i = box[0], j = box[1], k = box[2];
    const bool tf = (((int)i + (int)j + (int)k) & 1) != 0;
    const bool t1 = tet == 1, t2 = tet == 2, t3 = tet == 3, t4 = tet == 4;
    const bool b1 = tf ? !t4 : t1, b2 = tf ? !t3 : t2, b3 = tf ? t1 : !t3, b4 = tf ? t2 : !t4;
    const double e = 4.0 * g.eps;
    k1 = (k - i - j - (tf ? 1.0 : 0.0)) + (b1 ? e : -e);
    k2 = (k + i + j + (tf ? 1.0 : 2.0)) + (b2 ? e : -e);
    k3 = (k + i - j + (tf ? 1.0 : 0.0)) + (b3 ? e : -e);
    k4 = (k - i + j + (tf ? 1.0 : 0.0)) + (b4 ? e : -e);
    a1 = ballot(b1);
    a2 = ballot(b2);
    a3 = ballot(b3);
    a4 = ballot(b4);
    const bool mid = tet == 0;  // no side
    const bool ux = !mid & (tf ? t1 | t4 : t2 | t4), uy = !mid & (tf ? t2 | t4 : t2 | t3), uz = t1 | t2;
    const double w = -0.5 * g.eps;  // a wall's bound is moved out
    fx = mid ? -__DBL_MAX__ : (ux ? i + 1.0 - (i < ni ? e : w) : i + (i > 0.0 ? e : w)) * g.inc_x;
    fy = mid ? -__DBL_MAX__ : (uy ? j + 1.0 - (j < nj ? e : w) : j + (j > 0.0 ? e : w)) * g.inc_y;
    fz = mid ? -__DBL_MAX__ : (uz ? k + 1.0 - e : k + (k > 0.0 ? e : w)) * g.inc_z;
    lx = ballot(!ux);
    ly = ballot(!uy);
    lz = ballot(!uz);
    zmax = dmin(((double)g.nC2 - e) * g.inc_z, g.top_z - e * g.inc_z);
  }
  __device__ __forceinline__ uint64_t inside(const double* q, const Geom& g) const {
    const double ty = q[1] * g.rinc_y;
    const double s = __builtin_fma(q[0], g.rinc_x, ty), d = __builtin_fma(q[0], g.rinc_x, -ty);
    const double d1 = __builtin_fma(q[2], g.rinc_z, -s), d2 = __builtin_fma(q[2], g.rinc_z, s);
    const double d3 = __builtin_fma(q[2], g.rinc_z, d), d4 = __builtin_fma(q[2], g.rinc_z, -d);
    return ~((lanes_gt(d1, k1) ^ a1) | (lanes_gt(d2, k2) ^ a2) | (lanes_gt(d3, k3) ^ a3) | (lanes_gt(d4, k4) ^ a4) |
             (lanes_gt(q[0], fx) ^ lx) | (lanes_gt(q[1], fy) ^ ly) | (lanes_gt(q[2], fz) ^ lz)) &
           lanes_lt(q[2], zmax) & lanes_lt(__builtin_fabs(d2), 0x1p30);
  }
};

// ----------------------------------------------------------------- trip
// One unit of the reference's step schedule for one point of a lane (all lanes of a wave in lockstep, whatever unit each is at):
//   k == 0: y = Trel_c [p;1]; if cell(y) == c accept, else start the RK2 redo
//           (k = nStepsODE; p and c unchanged)   (calc_2Dto2D.cu:389-401)
//   k >  0: one RK2 midpoint substep of A_c from p (solveODE, :179-194);
//           p = y, c = cell(y), k--.
// Both kinds of trip share the table read, the first affine product and the
// cell lookup, so lanes in different modes diverge only over the midpoint
// arithmetic.  (Measured on gfx950: evaluating the midpoint in every lane
// and selecting, or chaining several Trel proposals speculatively so their
// lookups overlap, are both slower than this.)
// Returns true when the step is complete (the caller advances t).
template <int DIM, int TESS, bool POW2, bool FAST = false, bool EARLY = true>
__device__ __forceinline__ bool trip(double* p, int& c, int& k, const double*& row, int& nfb, const double* Ttab,
                                     const double* Atab, double h, int nS, const Geom& g) {
  constexpr int NE = DIM * (DIM + 1);
  const bool fast = (k == 0);
  double y[DIM];
  affine<DIM>(y, row, p);
  if (!fast) {  // RK2 midpoint substep (solveODE, calc_2Dto2D.cu:182-194)
    // The reference's h * v / 2 is fl(h v) halved; (h / 2) * v rounds the
    // same real number h v / 2, and halving commutes with rounding, so the
    // two agree bit for bit unless |h v / 2| is subnormal (below 2^-1022).
    // A nonzero v = A [p; 1] is at least ~2^-53 of its largest term, so that
    // takes table entries near 1e-290.  One multiply per coordinate fewer.
    const double hh = h * 0.5;
    double m[DIM];
#pragma unroll
    for (int d = 0; d < DIM; d++) m[d] = p[d] + hh * y[d];
    affine<DIM>(y, row, m);
#pragma unroll
    for (int d = 0; d < DIM; d++) y[d] = p[d] + y[d] * h;
  }
  const int cy = cell_of<DIM, TESS, POW2, FAST, EARLY>(y, g);
  // (Measured on gfx950: the state update below written as selects instead
  // of branches ran 3-4 % slower here and 11 % slower for 256 registration
  // chains.)
  if (!fast) {
#pragma unroll
    for (int d = 0; d < DIM; d++) p[d] = y[d];
    const bool done = --k == 0;
    row = (done ? Ttab : Atab) + mul24(cy, NE);  // (the same row when the cell did not change)
    c = cy;
    return done;
  }
  if (cy == c) {
#pragma unroll
    for (int d = 0; d < DIM; d++) p[d] = y[d];
    return true;
  }
  nfb++;
  if (nS > 0) {
    k = nS;
    row = Atab + mul24(c, NE);
    return false;
  }
  return true;  // zero substeps: the step leaves p where it was
}

// -------------------------------------------------------------- advance
// Integrates the calling lanes (t < tb on each that has a point) to step tb by
// the reference's schedule (calc_2Dto2D.cu:385-402: every step the Trel
// proposal, and when it leaves the cell nS RK2 substeps instead), in two phases
// taken in turn:
//
//   stretch  every lane whose point is in its cell by the bounds takes Trel
//            steps, its row and bounds in registers, until its point leaves
//            them or kSeg steps are done: nothing is looked up and no table
//            is read, because the cell does not change.
//   redo     the lanes that left look their proposal up: most left the cell
//            and run the step's nS RK2 substeps, all of them together; some
//            were only beside a facet and accept it.
//
// or, for coarse integrations (lockstep_pays), in lockstep (advance_lockstep):
// one proposal or substep of every lane at a time, its cell looked up and its
// row read each time (`trip`).
//
// Per point the sequence of IEEE operations is the reference's.
//
// What bounds calc_T is instruction issue: a wave alone on its SIMD issues an
// FP64 operation every 8 cycles, dependent or not, several waves one every 4;
// a launch of few waves ends with its slowest one.  A step of a stretch is 24
// VALU and 9 scalar instructions (2D type I: 8 the affine product, 8 the
// bounds, 8 the update) against 36 and 20 and LDS latency for a trip in
// lockstep, or 52 when some lane of the wave is at a redone step.  The loop has
// no divergent branch: lanes that have left stay where they are by selects.  A
// redo costs about as much as 20 steps of a stretch however many lanes share
// it, and a lane that waits for company delays the wave's end: hence kSeg (16,
// 24, 32 and 100 steps: 2D 2 000 000 points 534, 470, 448 us; 3D volume warp
// 351, 319, 308, 341 us).  On MI355X, lockstep -> phases: 2D random points,
// 1 000: 51 -> 41 us, 65 536: 56 -> 45, 2 000 000: 606 -> 430; grids, 512 x
// 512: 67 -> 67 (its slowest waves cross many facets), 2048 x 2048: 735 -> 580;
// 640 x 480 with fields that leave the image 175 -> 137; 1D, 10^6 points of 50
// cells 274 -> 195; 3D, 64 x 80 x 96 volume 331 -> 308.
//
// more: the caller has further points for lanes that finish; then it returns
// as soon as `refill` lanes have.
constexpr int kSeg = 32;
constexpr int kSegTraj = 12;  // calc_trajectory: lanes far apart in steps store to as many rows (16: +3 %, 8: +6 %)
// calc_trajectory, more rows than the 256 MiB cache holds: the steps that a lane
// may be ahead of its wave's last.  Rows are written a point at a time, so a
// line stays in a cache until the wave's lanes have all been there, and a lane
// falls behind by a segment whenever it changes cell.  100 000 points, 1 000
// steps of 1 substep (1.6 GB), no bound / 64 / 32 / 16 steps: 1D, 50 cells 958,
// 726, 375, 243 us (in lockstep 439); 2D, 500 steps of 3 431, 441, 391, 230
// (349).  500 000 2D points, 100 steps of 10: 494 -> 376 us.
constexpr int kSpread = 16;
constexpr int64_t kCacheBytes = 256 << 20;
constexpr int kRefill = 8;
constexpr int kTrips = 2;  // trips in lockstep between two looks at the lanes that are done (1: 8 % slower; 4: the same)

// Lockstep instead of phases for integrations of few large steps: points leave
// their cells every few of them, so a stretch is short, and every lane waits for
// the redo of whichever left.  Up to 100 substeps in all, phases -> lockstep,
// 100 000 points: 30 steps of 3, 2D 42 -> 29 us, 3D 60 -> 39; 100 steps of 1,
// 16 x 16 cells and a fast field 206 -> 95.  In 3D below 64 steps whatever the
// substeps, as more of a wave's points leave at each step there: grids of
// 262 144 points, 4 x 4 x 4 boxes, 20 steps of 100 938 -> 500 us, 30 of 10 134 ->
// 91 (random points within 16 % either way).  Beyond both, phases: 1D and 2D in
// 30 steps of 10 take 0.60 of the time of an older lockstep kernel (median of
// 36 calls), lockstep 0.73; 100 steps of 4 0.63 and 0.75.
__host__ __device__ constexpr bool lockstep_pays(int dim, int nT, int nS) {
  return (int64_t)nT * (nS > 0 ? nS : 1) <= 100 || (dim == 3 && nT < 64);
}

// The point at the domain's corner (0, 0).  With zero velocity on the walls
// its velocity is zero up to rounding: it drifts ~1e-16 out of the domain and
// with some fields flips between triangles 0 and 3 of box (0, 0) at every
// substep, so up to all its steps are redone, one dependent chain of 1 100
// units where its neighbours have ~110, and the wave (a launch of 512 x 512
// grid points: all of it) waits for it.  Alone in its wave it runs here to
// step tb: the two triangles' rows stay in registers, and the lookup is a few
// products and comparisons while the point is within an eighth of a box of
// the corner, where the reference's rules (calc_2Dto2D.cu:60-110) come down
// to: left of the corner (px <= 0) triangle 3 unless sy < sx, else 3 where
// sx < sy and 0 elsewhere (1 - x < y holds for no point this near).  So 3
// where sx < sy and 0 where sy < sx: the substeps' loop asks no more and
// leaves a tie or a point further out to `cell`.  It is one dependent chain
// of a lone wave, ~270 cycles a substep (570 with the whole rule and
// a branch per triangle in it): a 512 x 512 grid with a flipping corner 264 ->
// 195 us, the adjoint of 16 pairs of 128 x 128 (its forward sweep) 490 -> 380.
// Returns where it has left that neighbourhood.
// The caller's hooks: proposed(cell, cell of the proposal), substep(cell it
// starts in), done(step, cell, redone, start point, end point).
template <class Proposed, class Substep, class Done>
__device__ __forceinline__ void corner_steps(double* p, int& c, int& t, int tb, const double* Ttab,
                                             const double* Atab, double h, int nS, const Geom& g, Proposed proposed,
                                             Substep on_substep, Done done) {
  const double hh = h * 0.5, mx = 0.125 * g.inc_x, my = 0.125 * g.inc_y;
  double A0[6], A3[6];
#pragma unroll
  for (int e = 0; e < 6; e++) {
    A0[e] = Atab[e];
    A3[e] = Atab[18 + e];
  }
  // The cell of q, wave-uniform as there is one lane (its branches are then
  // scalar ones); `near` false: looked up, the point is not beside the corner.
  auto cell = [&](const double* q, bool& near) {
    near = (lanes_lt(__builtin_fabs(q[0]), mx) & lanes_lt(__builtin_fabs(q[1]), my)) != 0;
    if (!near) return (int)__builtin_amdgcn_readfirstlane(cell2<TESS_I, true>(q, g));
    const double sx = q[0] * g.rinc_x, sy = q[1] * g.rinc_y;
    const uint64_t left = lanes_lt(sx, sy) | (~lanes_gt(q[0], 0.0) & ~lanes_lt(sy, sx) & __builtin_amdgcn_read_exec());
    return left != 0 ? 3 : 0;
  };
  auto substep = [&](const double* A) {
    double y[2], m[2];
    affine<2>(y, A, p);
    m[0] = p[0] + hh * y[0];
    m[1] = p[1] + hh * y[1];
    affine<2>(y, A, m);
    p[0] = p[0] + y[0] * h;
    p[1] = p[1] + y[1] * h;
  };
  bool near = true;
  int cu = __builtin_amdgcn_readfirstlane(c);
  const int te = __builtin_amdgcn_readfirstlane(tb);
  int tu = __builtin_amdgcn_readfirstlane(t);
  while (near && tu < te) {
    const double q[2] = {p[0], p[1]};
    const int cq = cu;
    double y[2];
    affine<2>(y, Ttab + cu * 6, p);
    const int cy = cell(y, near);
    proposed(cu, cy);
    const bool redo = cy != cu;
    if (!redo) {
      p[0] = y[0];
      p[1] = y[1];
    } else {
      near = true;
      int s = nS;
      while (s > 0 && near) {
        uint64_t plain;  // beyond doubt: within a sixteenth of a box and on one side
        do {
          on_substep(cu);
          if (cu == 3) substep(A3);
          else substep(A0);
          const double sx = p[0] * g.rinc_x, sy = p[1] * g.rinc_y;
          const uint64_t lt = lanes_lt(sx, sy);
          plain = (lt | lanes_lt(sy, sx)) & lanes_lt(__builtin_fmax(__builtin_fabs(sx), __builtin_fabs(sy)), 0.0625);
          cu = lt != 0 ? 3 : 0;
          s--;
        } while (s > 0 && plain != 0);
        if (plain == 0) cu = cell(p, near);
      }
      for (; s > 0; s--) {  // (it has left: the step's other substeps)
        on_substep(cu);
        substep(Atab + cu * 6);
        cu = __builtin_amdgcn_readfirstlane(cell2<TESS_I, true>(p, g));
      }
    }
    done(tu, cq, redo, q, p);
    tu++;
  }
  c = cu;
  t = tu;
}

template <int DIM, int TESS, bool POW2, int MODE>
__device__ __forceinline__ void advance(double* p, int& c, int& t, int tb, int& nfb, const double* Ttab,
                                        const double* Atab, double h, int nS, const Geom& g, bool more_,
                                        int refill, double* __restrict__ traj, int64_t nPts, bool far) {
  constexpr int NE = DIM * (DIM + 1);
  // The reference's h * v / 2 is fl(h v) halved; (h / 2) * v rounds the same
  // real number h v / 2, and halving commutes with rounding, so the two agree
  // bit for bit unless |h v / 2| is subnormal (below 2^-1022).  A nonzero
  // v = A [p; 1] is at least ~2^-53 of its largest term, so that takes table
  // entries near 1e-290.  One multiply per coordinate fewer.
  const double hh = h * 0.5;
  const int nAll = __popcll(__builtin_amdgcn_read_exec());
  constexpr int seg = MODE == 1 ? kSegTraj : kSeg;
  const bool more = __builtin_amdgcn_readfirstlane((int)more_) != 0;  // (wave-uniform: kept in scalar registers)
  int cool = 0;  // rounds without a stretch (wave-uniform)
  for (;;) {
    const uint64_t todo = ballot(t < tb);
    const int nTodo = __popcll(todo);
    if (nTodo == 0 || (more && nAll - nTodo >= refill)) break;
    bool waits = t < tb;  // the lane takes part in the redo phase
    if (DIM == 2 && TESS == TESS_I && POW2 && nTodo == 1 && cool > 0) {  // one lane left, and no stretch for it
      if (waits && (c == 0 || c == 3) && __builtin_fabs(p[0]) < 0.125 * g.inc_x &&
          __builtin_fabs(p[1]) < 0.125 * g.inc_y) {
        corner_steps(
            p, c, t, tb, Ttab, Atab, h, nS, g, [](int, int) {}, [](int) {},
            [&](int step, int, bool redo, const double*, const double* q) {
              nfb += redo ? 1 : 0;
              if (MODE == 1) store_pt<2>(traj, (int64_t)step * nPts, q);
            });
        waits = false;
      }
    }
    if (cool > 0) {
      cool--;
    } else {
      CellBounds<DIM, TESS> B;
      double R[NE];
      const double* row = Ttab + mul24(c, NE);
#pragma unroll
      for (int e = 0; e < NE; e++) R[e] = row[e];
      B.enter(c, g);
      uint64_t go = B.inside(p, g) & todo;  // the lanes of the stretch
      if (go == 0) cool = 8;
      for (;;) {
        int lim = tb - t < seg ? tb : t + seg;
        if (MODE == 1 && far) {  // (uniform; every lane of the wave is here, those without a point at t >= tb)
          int m = t;
#pragma unroll
          for (int o = 32; o > 0; o >>= 1) {
            const int x = __shfl_xor(m, o, 64);
            m = x < m ? x : m;
          }
          lim = lim < m + kSpread ? lim : m + kSpread;
        }
        while (go != 0) {
          double y[DIM];
          affine<DIM>(y, R, p);
          go &= B.inside(y, g) & lanes_lt(t, lim);
          const bool in = lane_in(go);
#pragma unroll
          for (int d = 0; d < DIM; d++) p[d] = in ? y[d] : p[d];
          if (MODE == 1 && in) store_pt<DIM>(traj, (int64_t)t * nPts, p);
          t += in ? 1 : 0;
        }
        waits = t < lim;
        go = ballot(t < tb);  // with no lane waiting the cells are still the same
        if (go == 0 || ballot(waits) != 0 || (more && nAll - __popcll(go) >= refill)) break;
      }
    }
    if (waits) {
      const double* row = Ttab + mul24(c, NE);
      double y[DIM];
      affine<DIM>(y, row, p);
      const int cy = cell_of<DIM, TESS, POW2, true>(y, g);
      if (cy == c) {
#pragma unroll
        for (int d = 0; d < DIM; d++) p[d] = y[d];
      } else {
        nfb++;
        for (int s = 0; s < nS; s++) {
          row = Atab + mul24(c, NE);
          affine<DIM>(y, row, p);
          double m[DIM];
#pragma unroll
          for (int d = 0; d < DIM; d++) m[d] = p[d] + hh * y[d];
          affine<DIM>(y, row, m);
#pragma unroll
          for (int d = 0; d < DIM; d++) p[d] = p[d] + y[d] * h;
          c = cell_of<DIM, TESS, POW2, true>(p, g);
        }
      }
      if (MODE == 1) store_pt<DIM>(traj, (int64_t)t * nPts, p);
      t++;
    }
  }
}

// The same in lockstep.  k: substeps that a lane has to go in its step (0
// between steps), kept from call to call.  Every lane of the wave calls it, those
// without a point with t >= tb.
template <int DIM, int TESS, bool POW2, int MODE>
__device__ __forceinline__ void advance_lockstep(double* p, int& c, int& k, int& t, int tb, int& nfb,
                                                 const double* Ttab, const double* Atab, double h, int nS,
                                                 const Geom& g, bool more, int refill, double* __restrict__ traj,
                                                 int64_t nPts) {
  constexpr int NE = DIM * (DIM + 1);
  const double* row = (k == 0 ? Ttab : Atab) + mul24(c, NE);
  for (;;) {
    const int nTodo = __popcll(ballot(t < tb));
    if (nTodo == 0 || (more && 64 - nTodo >= refill)) break;
    for (int u = 0; u < kTrips; u++) {
      if (t < tb) {
        if (trip<DIM, TESS, POW2, true>(p, c, k, row, nfb, Ttab, Atab, h, nS, g)) {
          if (MODE == 1) store_pt<DIM>(traj, (int64_t)t * nPts, p);
          t++;
        }
      }
    }
  }
}

// --------------------------------------------------------- integration
// MODE 0: calc_T (write the end point).  MODE 1: calc_trajectory (write the
// point after every step into traj[(t*nPts + i)*DIM]).
//
// Lane state: p (current point), c (cell of p), t (steps done).  solveODE
// recomputes cell(p) at the top of every substep; here it is the lookup at
// the end of the previous one, of the same p: same value.  Lanes retire and
// take the next points of the block's range between calls of `advance`.
//
// Processing index i -> point index of n points that form a row-major grid
// of row length w: bands of r = 1 << lr rows are walked in tiles of r rows and
// 64 / r columns (64 consecutive indices one tile; w a multiple of 64 / r);
// what follows the last whole band, from nTiled on, maps to itself.  A
// bijection of [0, n) whatever w is.
struct GridOrder {
  int w = 0, lr = 3;   // w == 0: index order
  int64_t nTiled = 0;
  __device__ __forceinline__ int64_t operator()(int64_t i) const {
    if (i >= nTiled) return i;
    const int64_t t = i >> 6;
    const int u = (int)(i & 63), lc = 6 - lr, tpr = w >> lc;
    const int64_t ty = t / tpr;
    const int tx = (int)(t - ty * tpr);
    return ((ty << lr) + (u >> lc)) * (int64_t)w + (tx << lc) + (u & ((1 << lc) - 1));
  }
};

// 2D and 3D points that look like a row-major grid (of rows along x) are taken
// in tiles of x and y: neighbouring points flow alike and cross facets at about the same steps, so a wave's
// lanes need similar numbers of steps.  The row length is the first index, a
// multiple of 8 up to 8 x blockDim.x, where y changes from point 0's.  Only
// the processing order depends on it (every point's result is its own), so a
// wrong guess costs time only.  In two parts, so that the loads' latency
// passes while the tables are staged; barriers lie between the parts and
// after the first store to *w.  On MI355X: 512 x 512 points 80.4 -> 77.1 us in
// lockstep trips; 3D, 64 x 80 x 96 volume warp 314 -> 292 us (8 x 8 x 1 tiles
// instead of 64 points of a row).
template <int DIM>
struct RowProbe {
  double y0 = 0.0, yc = 0.0, yp = 0.0;
  __device__ __forceinline__ void load(const double* __restrict__ pts, int64_t n) {
    const int64_t i = 8 * ((int64_t)threadIdx.x + 1);
    if (i < n) {
      y0 = pts[1];
      yc = pts[i * DIM + 1];
      yp = pts[(i - 1) * DIM + 1];
    }
  }
  __device__ __forceinline__ void vote(int64_t n, int* w) const {
    const int64_t i = 8 * ((int64_t)threadIdx.x + 1);
    if (i < n && yc != y0 && yp == y0) atomicMin(w, (int)i);
  }
};

__device__ __forceinline__ GridOrder grid_order(int w, int64_t n) {
  GridOrder o;
  if (w == 0x7fffffff) return o;
  while (o.lr > 0 && (((int64_t)w << o.lr) > n || (w & ((64 >> o.lr) - 1)) != 0)) o.lr--;
  if (o.lr == 0) return o;
  o.w = w;
  o.nTiled = n / ((int64_t)w << o.lr) * ((int64_t)w << o.lr);
  return o;
}

// The block's waves integrate the n points that follow `begin` in the
// processing order (indices into pos0, out and nfb_out; with gord.w > 0
// through it, counted from gbase, with lord through begin + lord[i], a tile's order held in LDS).
// They draw them from one cursor in LDS (zero at the call, behind a barrier):
// with a range for each wave the block waited for the one whose points cross
// the most facets (256 batched instances, 16 waves a block: 11.4 -> 9.6 ms).
// Block-uniform arguments; every lane of the block calls it.
//
// corner: a grid that starts beside the domain's corner has its first point
// integrated by a block of its own (2), and the block that it falls to leaves
// it out (1): it may be `corner_steps`'s, and among 63 neighbours it took one
// step to their stretch of 32 until they were done (512 x 512 grid with a
// flipping corner 195 -> 163 us; other launches, one block more, the same).
template <int DIM, int TESS, bool POW2, int MODE, bool LOCK>
__device__ __forceinline__ void integrate_points(int64_t begin, int n, int* cursor, const double* __restrict__ pos0,
                                                double* __restrict__ out, const double* Ttab, const double* Atab,
                                                double h, int nT, int nS, int64_t nPts, const Geom& g,
                                                int32_t* __restrict__ nfb_out, const GridOrder& gord,
                                                int64_t gbase, const uint16_t* lord, int corner) {
  // a grid's tiles are 64 neighbouring points that need similar work, so a
  // wave takes one after another (2048 x 2048 points: 750 -> 610 us); other
  // waves take the next points as soon as kRefill lanes are free (256 batched
  // instances, 8 instead of 16: 14.3 -> 13.9 ms, 32: 16.7; 64: 15.3).  Trajectories
  // larger than the cache: a wave's points all start together, or the others
  // would wait for the new ones (kSpread).
  const bool far = MODE == 1 && nT * nPts > kCacheBytes / (8 * DIM);
  const int refill = gord.w > 0 || far ? 64 : kRefill;
  double p[DIM];
#pragma unroll
  for (int d = 0; d < DIM; d++) p[d] = 0.0;
  int c = 0, k = 0, t = nT, nfb = 0;  // (an idle lane is at step nT)
  int64_t my = 0;
  bool active = false, more = true;
  int taken = 0;  // points the cursor leaves out
  if (DIM == 2 && TESS == TESS_I && POW2 && MODE == 0 && corner != 0) {
    bool near = false;
    if (gord.w > 0) {
      my = gbase + gord(begin - gbase);
      load_pt<DIM>(pos0, my, p);
      near = ballot(__builtin_fabs(p[0]) < 0.125 * g.inc_x && __builtin_fabs(p[1]) < 0.125 * g.inc_y) != 0;
    }
    if (corner == 2) {
      if (!near) return;
      active = threadIdx.x == 0;
      more = false;
      t = active ? 0 : nT;
      c = cell_of<DIM, TESS, POW2>(p, g);
    }
    taken = near ? 1 : 0;
  }
  for (;;) {
    if (active && t >= nT) {  // retire a finished point
      if (MODE == 0) store_pt<DIM>(out, my, p);
      if (nfb_out) nfb_out[my] = nfb;
      active = false;
    }
    const uint64_t idle = ballot(!active);
    if (idle != 0 && more) {  // idle lanes take the next points
      int next = 0;
      if (lane_id() == 0) next = atomicAdd(cursor, __popcll(idle));
      next = __builtin_amdgcn_readfirstlane(next);
      if (!active) {
        const int cand = next + taken + rank_in(idle);
        if (cand < n) {
          my = gord.w > 0 ? gbase + gord(begin - gbase + cand) : begin + (lord ? (int)lord[cand] : cand);
          active = true;
          load_pt<DIM>(pos0, my, p);
          c = cell_of<DIM, TESS, POW2>(p, g);
          t = 0;
          nfb = 0;
        }
      }
      more = next + taken + __popcll(idle) < n;
    }
    if (ballot(active) == 0) break;
    if (LOCK) {
      advance_lockstep<DIM, TESS, POW2, MODE>(p, c, k, t, nT, nfb, Ttab, Atab, h, nS, g, more, refill,
                                              MODE == 1 ? out + my * DIM : nullptr, nPts);
    } else if (MODE == 1 || (active && t < nT)) {  // (calc_trajectory's compares the lanes' steps: all of them call it)
      advance<DIM, TESS, POW2, MODE>(p, c, t, nT, nfb, Ttab, Atab, h, nS, g, more, refill,
                                     MODE == 1 ? out + my * DIM : nullptr, nPts, far);
    }
  }
}

// (Two copies of the loop: phases and lockstep in one, chosen wave by wave as
// points left the bounds of their cells, cost the phases 2-10 %, and up to 30 %
// where a wave's last lane redoes its steps.)
template <int DIM, int TESS, bool POW2, int MODE>
__device__ __forceinline__ void integrate_range(int64_t begin, int n, int* cursor, const double* __restrict__ pos0,
                                                double* __restrict__ out, const double* Ttab, const double* Atab,
                                                double h, int nT, int nS, int64_t nPts, const Geom& g,
                                                int32_t* __restrict__ nfb_out, const GridOrder& gord = GridOrder(),
                                                int64_t gbase = 0, const uint16_t* lord = nullptr,
                                                int corner = 0) {
  if (lockstep_pays(DIM, nT, nS))  // (kernel arguments: uniform)
    integrate_points<DIM, TESS, POW2, MODE, true>(begin, n, cursor, pos0, out, Ttab, Atab, h, nT, nS, nPts, g, nfb_out,
                                                  gord, gbase, lord, corner);
  else
    integrate_points<DIM, TESS, POW2, MODE, false>(begin, n, cursor, pos0, out, Ttab, Atab, h, nT, nS, nPts, g, nfb_out,
                                                   gord, gbase, lord, corner);
}

// Launches of k_integrate that may have a block ahead of the points' own, for
// the corner's point (the cases of `corner_steps`).
constexpr bool has_corner_block(int dim, int tess, bool pow2, int mode) {
  return mode == 0 && dim == 2 && tess == TESS_I && pow2;
}

// The fewest steps for which a grid's points are taken in tiles: for 1 to 3 the
// order gains less than the look at the points costs (one step, 262 144 points
// in 3D: 11.0 us, with it 13.1).
constexpr int kOrderSteps = 4;

// LDS that the integration kernels hold besides their tables and orders (the
// cursors, a run's row length): a launch's dynamic LDS leaves room for it.
constexpr int kOwnLds = 16;

template <int DIM, int TESS, bool POW2, bool LDS, int MODE>
__global__ void __launch_bounds__(1024) __attribute__((amdgpu_waves_per_eu(5)))
    k_integrate(const double* __restrict__ pos0, double* __restrict__ out,
                const double* __restrict__ Trels, const double* __restrict__ As, double h,
                int nT, int nS, int64_t nPts, Geom g, int nC, int ptsPerWave,
                int32_t* __restrict__ nfb_out, PrepSrc ps, int corner) {
  constexpr int NE = DIM * (DIM + 1);
  extern __shared__ double lds[];
  __shared__ int grid_w, cursor;
  const bool detect = MODE == 0 && DIM > 1 && nT >= kOrderSteps;
  const bool own = has_corner_block(DIM, TESS, POW2, MODE) && corner != 0;  // block 0 is the corner's
  RowProbe<DIM> probe;
  if (threadIdx.x == 0) {
    grid_w = 0x7fffffff;
    cursor = 0;
  }
  if (detect) probe.load(pos0, nPts);
  __syncthreads();
  const double* Ttab = Trels;
  const double* Atab = As;
  if (LDS) {
    if (ps.raw) stage_tables_prep<DIM>(lds, ps, nC);  // (a kernel argument: uniform)
    else stage_tables<NE>(lds, Trels, As, nC);
    Ttab = lds;
    Atab = lds + nC * NE;
  }
  GridOrder gord;
  if (detect) {
    probe.vote(nPts, &grid_w);
    __syncthreads();
    gord = grid_order(grid_w, nPts);
  }
  const int per = (int)(blockDim.x >> 6) * ptsPerWave;
  const int64_t blk = own ? (blockIdx.x == 0 ? 0 : (int64_t)blockIdx.x - 1) : (int64_t)blockIdx.x;
  const int64_t begin = blk * per;
  const int n = nPts - begin < per ? (int)(nPts - begin) : per;
  integrate_range<DIM, TESS, POW2, MODE>(begin, n, &cursor, pos0, out, Ttab, Atab, h, nT, nS, nPts, g, nfb_out, gord, 0,
                                         nullptr, !own ? 0 : blockIdx.x == 0 ? 2 : blockIdx.x == 1 ? 1 : 0);
}

// ---------------------------------------------------------- sensitivity
// calc_grad_theta (cpab/gpu/calc_2Dto2D.cu:202-319, 448-491): calc_T_simple
// together with the forward sensitivity q_j = dp/dtheta_j of every basis
// column j, integrated by the same RK2 (q' = B_j [p;1] + A_lin q).  Grid
// (point blocks, column chunks): a thread owns one point and JC columns; the
// reference keeps q in global memory and re-reads it every substep, here it
// stays in registers (same values), and so do the cell's row and the columns'
// basis rows (layout (d, nC, DIM, DIM+1)), read again when the point has left
// the cell.  Output grad (nPts, DIM, d) and, from the first chunk, the end
// points.  The last chunk ends at column d: it repeats columns of the one
// before where JC does not divide d (the same values).
//
// Bound by FP64 instructions without FMA, 38 a substep and column and 48 a
// substep; no branch between the columns, whose LDS reads each stalled the
// wave when the rows were read every substep (and staged: now a wave reads
// rows on the ~1/4 of its substeps in which some point changes cell, and from
// LDS that measured the same).  128 x 128 grid, 62 columns: 1.86 -> 1.55 ms
// (0.25 of it the corner's pixel, which changes cell every substep); 16 384
// random points 2.79 -> 1.35 ms (28 T instructions/s of the 39 that two waves
// a SIMD can issue), 2 000: 1.55 -> 0.30, 500: 1.55 -> 0.20.
template <int DIM, int TESS, bool POW2, int JC>
__global__ void __launch_bounds__(256, 2)
    k_grad_theta(const double* __restrict__ pos0, double* __restrict__ pos, const double* __restrict__ As,
                 const double* __restrict__ Bs, double* __restrict__ grad, int d, double h, int nSteps,
                 int64_t nPts, Geom g, int nC) {
  constexpr int NE = DIM * (DIM + 1);
  const int64_t jc = ((int64_t)blockIdx.z * gridDim.y + blockIdx.y) * JC;
  if (jc >= d) return;
  const int j0 = jc + JC <= d ? (int)jc : (d > JC ? d - JC : 0);
  const int nj = d < JC ? d : JC;
  const double* Bl = Bs + (int64_t)j0 * nC * NE;
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= nPts) return;
  const double hh = h * 0.5;  // (as in `advance`)
  double p[DIM], q[JC][DIM], A[NE], B[JC][NE];
#pragma unroll
  for (int jj = 0; jj < JC; jj++)
#pragma unroll
    for (int i = 0; i < DIM; i++) q[jj][i] = 0.0;
  load_pt<DIM>(pos0, idx, p);
  CellBounds<DIM, TESS> bounds;
  const uint64_t all = __builtin_amdgcn_read_exec();
  uint64_t in = 0;  // lanes whose point is in the cell of their rows
  int c = -1;
  for (int s = 0; s < nSteps; s++) {
    if (in != all) {
      if (!lane_in(in)) {
        const int cn = cell_of<DIM, TESS, POW2>(p, g);
        if (cn != c) {
          c = cn;
#pragma unroll
          for (int e = 0; e < NE; e++) A[e] = As[c * NE + e];
#pragma unroll
          for (int jj = 0; jj < JC; jj++)
#pragma unroll
            for (int e = 0; e < NE; e++) B[jj][e] = Bl[((jj < nj ? jj : 0) * nC + c) * NE + e];
        }
      }
      bounds.enter(c, g);
    }
    double v[DIM], pMid[DIM];
    affine<DIM>(v, A, p);
#pragma unroll
    for (int i = 0; i < DIM; i++) pMid[i] = p[i] + hh * v[i];
    affine<DIM>(v, A, pMid);
#pragma unroll
    for (int jj = 0; jj < JC; jj++) {
      double BtT[DIM], AdT[DIM], qMid[DIM];
      affine<DIM>(BtT, B[jj], p);
      linear<DIM>(AdT, A, q[jj]);
#pragma unroll
      for (int i = 0; i < DIM; i++) qMid[i] = q[jj][i] + hh * (BtT[i] + AdT[i]);
      affine<DIM>(BtT, B[jj], pMid);
      linear<DIM>(AdT, A, qMid);
#pragma unroll
      for (int i = 0; i < DIM; i++) q[jj][i] += (BtT[i] + AdT[i]) * h;
    }
#pragma unroll
    for (int i = 0; i < DIM; i++) p[i] += v[i] * h;
    in = bounds.inside(p, g);
  }
  if (jc == 0) store_pt<DIM>(pos, idx, p);
#pragma unroll
  for (int jj = 0; jj < JC; jj++)
    if (jj < nj)
#pragma unroll
      for (int i = 0; i < DIM; i++) grad[(idx * DIM + i) * d + j0 + jj] = q[jj][i];
}

// calc_T_simple: nStepsODE * nTimeSteps RK2 substeps (calc_2Dto2D.cu:412-445),
// with a lookup only where some point of the wave has left the bounds of its
// cell.  Bound by FP64 instructions: 35 a substep and point and 12 for the
// bounds' test, against 75 and a table read with a lookup in each substep; but
// to look up and form the bounds is 80.  Waves that gain nothing by bounds have
// some point outside them nearly always (points on walls and corners, 64
// random points in a coarse integration): after three stretches in a row that
// ended at once (one or two in a coarse integration, where short ones are the
// rule) come 3, 7, .. 63 substeps with a lookup each before the next one.
// MI355X, 1 000 substeps, lookups in each / bounds always / this: 2D type I,
// 100 000 random points 303 / 200 / 207 us, 256 x 256 grid 263 / 347 / 197,
// 3 x 5 cells 738 / 207 / 209; 3D, 65 536 point grid 414 / 734 / 333; 1D,
// 1 000 points 226 / 80 / 82.  100 substeps: 2D, 100 000 points 33 / 45 / 35.
template <int DIM, int TESS, bool POW2, bool LDS>
__global__ void __launch_bounds__(1024)
    k_simple(const double* __restrict__ pos0, double* __restrict__ out, const double* __restrict__ As,
             double h, int nSteps, int64_t nPts, Geom g, int nC) {
  constexpr int NE = DIM * (DIM + 1);
  extern __shared__ double lds[];
  const double* Atab = As;
  if (LDS) {
    for (int i = threadIdx.x; i < nC * NE; i += blockDim.x) lds[i] = As[i];
    __syncthreads();
    Atab = lds;
  }
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nPts) return;
  const double hh = h * 0.5;  // (as in `advance`)
  double p[DIM], A[NE];
  load_pt<DIM>(pos0, i, p);
  auto lookup = [&]() {
    const int c = cell_of<DIM, TESS, POW2>(p, g);
#pragma unroll
    for (int e = 0; e < NE; e++) A[e] = Atab[c * NE + e];
    return c;
  };
  auto substep = [&]() {
    double y[DIM], m[DIM];
    affine<DIM>(y, A, p);
#pragma unroll
    for (int d = 0; d < DIM; d++) m[d] = p[d] + hh * y[d];
    affine<DIM>(y, A, m);
#pragma unroll
    for (int d = 0; d < DIM; d++) p[d] += y[d] * h;
  };
  const uint64_t all = __builtin_amdgcn_read_exec();
  const bool coarse = nSteps <= 128;  // (few substeps in all are large ones)
  const int kShort = TESS == TESS_I && coarse ? 2 : 1;
  CellBounds<DIM, TESS> bounds;
  uint64_t in = 0;  // lanes whose point is in the cell of their row
  // substeps left, those left at the last lookup, short stretches in a row (wave-uniform)
  int s = nSteps, last = nSteps, shorts = coarse ? 1 : -1;
  for (; s > 0; s--) {
    if (in != all) {
      shorts = last - s > kShort ? 0 : shorts + 1;
      if (shorts >= 3)
        for (int u = (1 << (shorts < 7 ? shorts - 1 : 6)) - 1; u > 0 && s > 1; u--, s--) {
          lookup();
          substep();
        }
      last = s;
      bounds.enter(lookup(), g);
    }
    substep();
    in = bounds.inside(p, g);
  }
  store_pt<DIM>(out, i, p);
}

// calc_v: bound by memory (one point read, one velocity written).  A block
// stages the table once and walks over the points; a block per 256 points
// staged a table of 1 024 cells (48 KiB) for 8 KiB of points.  On MI355X,
// 2048 x 2048 points: 1 024 cells 90.5 -> 24.1 us (5.6 TB/s), 64 cells 21.5 ->
// 21.7 us; two or four points loaded ahead in each thread measured the same.
template <int DIM, int TESS, bool POW2, bool LDS>
__global__ void __launch_bounds__(1024)
    k_velocity(const double* __restrict__ pts, double* __restrict__ vel, const double* __restrict__ As,
               int64_t nPts, Geom g, int nC) {
  constexpr int NE = DIM * (DIM + 1);
  extern __shared__ double lds[];
  const double* Atab = As;
  if (LDS) {
    for (int i = threadIdx.x; i < nC * NE; i += blockDim.x) lds[i] = As[i];
    __syncthreads();
    Atab = lds;
  }
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < nPts; i += stride) {
    double p[DIM], v[DIM];
    load_pt<DIM>(pts, i, p);
    affine<DIM>(v, Atab + cell_of<DIM, TESS, POW2>(p, g) * NE, p);
    store_pt<DIM>(vel, i, v);
  }
}

template <int DIM, int TESS, bool POW2>
__global__ void k_cell_idx(const double* __restrict__ pts, int32_t* __restrict__ cell, int64_t nPts, Geom g) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nPts) return;
  double p[DIM];
  load_pt<DIM>(pts, i, p);
  cell[i] = cell_of<DIM, TESS, POW2>(p, g);
}

// ---------------------------------------------------- remap + likelihood
// Bilinear sample, zero outside (OpenCV INTER_LINEAR, BORDER_CONSTANT 0),
// weights from the double coordinates' fractional parts, float arithmetic.
__device__ __forceinline__ float sample2(const float* __restrict__ img, int H, int W, double x, double y) {
  const double xf = floor(x), yf = floor(y);
  // a full pixel or more outside, or not a number: zero
  if (!(xf >= -1.0 && xf < (double)W && yf >= -1.0 && yf < (double)H)) return 0.f;
  const float fx = (float)(x - xf), fy = (float)(y - yf);
  float v00 = 0.f, v01 = 0.f, v10 = 0.f, v11 = 0.f;
  const int x0 = (int)xf, y0 = (int)yf, x1 = x0 + 1, y1 = y0 + 1;
  const bool okx0 = x0 >= 0, okx1 = x1 < W, oky0 = y0 >= 0, oky1 = y1 < H;
  if (oky0 && okx0) v00 = img[(int64_t)y0 * W + x0];
  if (oky0 && okx1) v01 = img[(int64_t)y0 * W + x1];
  if (oky1 && okx0) v10 = img[(int64_t)y1 * W + x0];
  if (oky1 && okx1) v11 = img[(int64_t)y1 * W + x1];
  const float gx = 1.f - fx, gy = 1.f - fy;
  const float a = gx * v00 + fx * v01;
  const float b = gx * v10 + fx * v11;
  return gy * a + fy * b;
}

__device__ __forceinline__ float sample3(const float* __restrict__ vol, int D, int H, int W, double x,
                                         double y, double z) {
  const double xf = floor(x), yf = floor(y), zf = floor(z);
  if (!(xf >= -1.0 && xf < (double)W && yf >= -1.0 && yf < (double)H && zf >= -1.0 && zf < (double)D))
    return 0.f;
  const float fx = (float)(x - xf), fy = (float)(y - yf), fz = (float)(z - zf);
  float v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  const int x0 = (int)xf, y0 = (int)yf, z0 = (int)zf;
#pragma unroll
  for (int dz = 0; dz < 2; dz++)
#pragma unroll
    for (int dy = 0; dy < 2; dy++)
#pragma unroll
      for (int dx = 0; dx < 2; dx++) {
        const int xx = x0 + dx, yy = y0 + dy, zz = z0 + dz;
        if (xx >= 0 && xx < W && yy >= 0 && yy < H && zz >= 0 && zz < D)
          v[dz * 4 + dy * 2 + dx] = vol[((int64_t)zz * H + yy) * W + xx];
      }
  const float gx = 1.f - fx, gy = 1.f - fy, gz = 1.f - fz;
  const float a0 = gx * v[0] + fx * v[1];
  const float a1 = gx * v[2] + fx * v[3];
  const float a2 = gx * v[4] + fx * v[5];
  const float a3 = gx * v[6] + fx * v[7];
  const float b0 = gy * a0 + fy * a1;
  const float b1 = gy * a2 + fy * a3;
  return gz * b0 + fz * b1;
}

__global__ void k_remap2d(const double* __restrict__ pts, const float* __restrict__ img,
                          float* __restrict__ out, int H, int W) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (int64_t)H * W) return;
  const double2 q = *reinterpret_cast<const double2*>(pts + 2 * i);
  out[i] = sample2(img, H, W, q.x, q.y);
}

__global__ void k_remap3d(const double* __restrict__ pts, const float* __restrict__ vol,
                          float* __restrict__ out, int D, int H, int W) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (int64_t)D * H * W) return;
  out[i] = sample3(vol, D, H, W, pts[3 * i], pts[3 * i + 1], pts[3 * i + 2]);
}

// Block sum of a per-lane double through LDS; result valid in thread 0.
__device__ __forceinline__ double block_sum(double v, double* red) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  const int w = threadIdx.x >> 6, nw = blockDim.x >> 6;
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[w] = v;
  __syncthreads();
  double s = 0.0;
  if (threadIdx.x == 0)
    for (int i = 0; i < nw; i++) s += red[i];
  return s;
}

// Per-block partial sums of (x - y)^2 over float images; the difference and
// its square are taken in double (two FP64 ops per pixel, and the sum of
// 10^5 terms keeps ~1e-15 relative accuracy instead of ~1e-7).
__global__ void k_ssd_partial(const float* __restrict__ x, const float* __restrict__ y, int64_t n,
                              double* __restrict__ partial) {
  __shared__ double red[16];
  double acc = 0.0;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    const double e = (double)x[i] - (double)y[i];
    acc += e * e;
  }
  const double s = block_sum(acc, red);
  if (threadIdx.x == 0) partial[blockIdx.x] = s;
}

// ll = -0.5 / sigma^2 * sum(partials), one wave (gaussian.py:30-34 + sum).
__global__ void k_reduce_ll(const double* __restrict__ partial, int n, double sigma, double* __restrict__ ll) {
  double acc = 0.0;
  for (int i = threadIdx.x; i < n; i += 64) acc += partial[i];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o, 64);
  if (threadIdx.x == 0) *ll = acc * (-0.5 / (sigma * sigma));
}

}  // namespace cpab
