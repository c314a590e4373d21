// Many independent calc_T problems in one persistent launch.
//
// Each instance has its own tessellation (cell counts, increments), its own
// tables (Trels then signed As, staged per instance in one table buffer) and
// its own point range in one concatenated point buffer.  The host cuts every
// instance into tiles of at most `tile` points (the largest first) and the
// kernel's blocks take up to `chunk` consecutive tiles at a time from a queue
// (one atomic per grab; a block leaves when the queue is exhausted, so every
// block ends).  A block keeps the tables of the instance it is working on in
// LDS and reloads them only when a tile of another instance comes; the waves
// of a block draw the tile's points from one cursor and integrate them with
// k_integrate's two phases (`advance`).  Per point the arithmetic is exactly calc_T's, so a
// point gives the same bits batched or alone.
#pragma once
#include "cpab_kernels.h"

#pragma clang fp contract(off)

namespace cpab {

struct BatchInst {
  Geom g;
  int nC;
  int pad;
  int64_t tab;   // offset (doubles) of the instance's tables: Trels (nC x NE), then signed As
  int64_t pts;   // offset (points) of the instance's first point
  int64_t nPts;
  int64_t cell;  // offset of the instance's first cell in the concatenated As input
};

struct BatchTile {
  int inst;
  int pad;
  int64_t begin, end;  // point range, absolute indices into the point buffer
};

// Signed As and Trels of every cell of every instance, into the table buffer.
// One lane per cell of the concatenated input As (cells in instance order).
template <int DIM>
__global__ void k_batch_prep(const BatchInst* __restrict__ insts, int nInst, const double* __restrict__ As,
                             int64_t nCells, int sign, double dt, double* __restrict__ tables, int p) {
  constexpr int NE = DIM * (DIM + 1);
  const int64_t cg = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (cg >= nCells) return;
  int lo = 0, hi = nInst - 1;  // the instance holding cell cg
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (insts[mid].cell <= cg) lo = mid;
    else hi = mid - 1;
  }
  const BatchInst& I = insts[lo];
  const int64_t c = cg - I.cell;
  double sA[NE], T[NE];
  prep_cell<DIM>(As + cg * NE, sign, dt, sA, T, p);
  double* Tt = tables + I.tab;
#pragma unroll
  for (int k = 0; k < NE; k++) {
    Tt[c * NE + k] = T[k];
    Tt[(int64_t)I.nC * NE + c * NE + k] = sA[k];
  }
}

__global__ void k_batch_reset(unsigned int* queue) {
  if (threadIdx.x == 0) *queue = 0u;
}

// Processing order of a tile's points by position: a counting sort of the
// tile's point indices over a grid of buckets on the domain (nb per axis, a
// power of two up to 1 024 in 1D, 32 in 2D, 8 in 3D, at least 16 points a
// bucket on average), buckets in row order, built in LDS by the whole block.
// Neighbouring points flow alike and cross facets at about the same steps,
// so a wave's lanes then need closer numbers of steps and redos than for
// points in input order.  Within a bucket the order follows the LDS atomics, which may
// differ from run to run: that changes which lane integrates a point and
// when, never the point's result.
constexpr int kBucketTileMax = 16384;  // the most points of a sorted tile (16-bit indices)
constexpr int kBucketMax = 1024;       // buckets
// The most points of a tile or an item taken at a time: a block's waves draw
// them from a 32-bit cursor, which each wave's last draw leaves up to 64 past
// the end (integrate_range's `next + taken + 64` is the largest sum).
constexpr int kItemMax = 1 << 30;
static_assert((int64_t)kItemMax + 64 * (1024 / 64) + 1 + 64 <= INT32_MAX, "integrate_range's cursor");

template <int DIM>
__device__ __forceinline__ int bucket_of(const double* p, const double* sc, int nb) {
  // (NaN coordinates go to a border bucket: fmin/fmax return the other operand)
  int b = 0;
#pragma unroll
  for (int d = DIM - 1; d >= 0; d--) b = b * nb + (int)fmax(0.0, fmin(p[d] * sc[d], (double)(nb - 1)));
  return b;
}

template <int DIM>
__device__ void tile_bucket_order(const double* __restrict__ pos0, int64_t begin, int n, const Geom& g,
                                  unsigned int* hist, uint16_t* idx) {
  constexpr int NBMAX = DIM == 1 ? 1024 : (DIM == 2 ? 32 : 8);
  int nb = 1, nbk = 1;
  while (nb < NBMAX && 16 * (nbk << DIM) <= n) {
    nb <<= 1;
    nbk <<= DIM;
  }
  double sc[DIM];
  sc[0] = (double)nb / ((double)g.nC0 * g.inc_x);
  if (DIM > 1) sc[DIM > 1 ? 1 : 0] = (double)nb / ((double)g.nC1 * g.inc_y);
  if (DIM > 2) sc[DIM > 2 ? 2 : 0] = (double)nb / ((double)g.nC2 * g.inc_z);
  __syncthreads();  // every wave is done with the previous tile's order
  for (int i = threadIdx.x; i < nbk; i += blockDim.x) hist[i] = 0u;
  __syncthreads();
  for (int j = threadIdx.x; j < n; j += blockDim.x) {
    double p[DIM];
    load_pt<DIM>(pos0, begin + j, p);
    atomicAdd(&hist[bucket_of<DIM>(p, sc, nb)], 1u);
  }
  __syncthreads();
  if (threadIdx.x < 64) {  // exclusive scan by the first wave, each lane a run of buckets
    const int per = (nbk + 63) >> 6;
    const int lo = (int)threadIdx.x * per;
    const int hi = lo + per < nbk ? lo + per : nbk;
    unsigned int sum = 0u;
    for (int i = lo; i < hi; i++) sum += hist[i];
    unsigned int x = sum;
    for (int d = 1; d < 64; d <<= 1) {
      const unsigned int y = __shfl_up(x, d, 64);
      if ((int)threadIdx.x >= d) x += y;
    }
    unsigned int run = x - sum;
    for (int i = lo; i < hi; i++) {
      const unsigned int c = hist[i];
      hist[i] = run;
      run += c;
    }
  }
  __syncthreads();
  for (int j = threadIdx.x; j < n; j += blockDim.x) {
    double p[DIM];
    load_pt<DIM>(pos0, begin + j, p);
    idx[atomicAdd(&hist[bucket_of<DIM>(p, sc, nb)], 1u)] = (uint16_t)j;
  }
  __syncthreads();
}

template <int DIM, int TESS, bool POW2>
__global__ void __launch_bounds__(1024)
    k_integrate_batch(const BatchInst* __restrict__ insts, const BatchTile* __restrict__ tiles, int nTiles, int chunk,
                      int least, unsigned int* __restrict__ queue, const double* __restrict__ tables,
                      const double* __restrict__ pos0, double* __restrict__ out, double h, int nT, int nS,
                      int32_t* __restrict__ nfb_out, int sort_off) {
  constexpr int NE = DIM * (DIM + 1);
  extern __shared__ double lds[];
  __shared__ int s_t0, s_t1, cursor;
  // sort_off > 0: the tiles' processing order by position, in LDS after
  // the tables (sort_off doubles in): bucket counters, then indices
  unsigned int* hist = reinterpret_cast<unsigned int*>(lds + sort_off);
  uint16_t* idx = reinterpret_cast<uint16_t*>(hist + kBucketMax);
  int cur = -1;  // instance whose tables are in LDS (block-uniform)
  for (;;) {
    __syncthreads();  // every wave is done with the previous chunk's s_t0
    if (threadIdx.x == 0) {
      // `chunk` tiles at a time while each block has four such grabs ahead of
      // it, then fewer, in the end `least` (256 instances, tiles of 16 384, chunk
      // 4: 2 400 tiles are 2.3 grabs for each of 256 blocks, and the launch
      // waited for those that took three)
      const unsigned int seen = __hip_atomic_load(queue, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      const int left = seen < (unsigned int)nTiles ? nTiles - (int)seen : 0;
      int k = left / (4 * (int)gridDim.x);
      k = k < least ? least : (k > chunk ? chunk : k);
      s_t0 = (int)atomicAdd(queue, (unsigned int)k);
      s_t1 = s_t0 + k;
    }
    __syncthreads();
    const int t0 = s_t0;
    if (t0 >= nTiles) break;
    const int t1 = s_t1 < nTiles ? s_t1 : nTiles;
    for (int t = t0; t < t1; t++) {
      const BatchTile tl = tiles[t];
      const int nC = insts[tl.inst].nC;
      if (tl.inst != cur) {
        const double* src = tables + insts[tl.inst].tab;
        __syncthreads();  // the previous tables are no longer read
        for (int i = threadIdx.x; i < 2 * nC * NE; i += blockDim.x) lds[i] = src[i];
        __syncthreads();
        cur = tl.inst;
      }
      const Geom g = insts[tl.inst].g;
      const int n = (int)(tl.end - tl.begin);
      const uint16_t* lord = nullptr;
      __syncthreads();  // every wave is done with the previous tile's points
      if (threadIdx.x == 0) cursor = 0;
      if (sort_off > 0 && n <= kBucketTileMax) {  // (block-uniform)
        tile_bucket_order<DIM>(pos0, tl.begin, n, g, hist, idx);
        lord = idx;
      } else {
        __syncthreads();
      }
      integrate_range<DIM, TESS, POW2, 0>(tl.begin, n, &cursor, pos0, out, lds, lds + nC * NE, h, nT, nS, 0, g, nfb_out,
                                          GridOrder(), 0, lord);
    }
  }
}

}  // namespace cpab

namespace cpab {

// A tile of one request of a served mix: its own tables, points and
// geometry, so a launch can take tiles of any set of requests.
struct WorkItem {
  Geom g;
  int nC;
  int pad;
  const double* trels;   // (nC, NE)
  const double* as;      // (nC, NE) signed As
  const double* pos0;
  double* out;
  int64_t begin, end;    // point range within the request's arrays
};

// Grabs: `chunk` items, or more while at least kGrabsAhead larger ones are
// ahead of each block.  Consecutive items of one request are taken together:
// an item of one point per lane kept its block waiting for its slowest wave,
// and several rows of a grid can be walked in tiles (RowProbe) where one row
// cannot.  The served mix, 48 requests waiting, on MI355X (launches of up to
// 2 048 items of 1 024 points): 2D 529 -> 427 us a launch, 3D 780 -> 707 us;
// runs of up to 3 or 8 items measured 461 and 480 us (2D).
constexpr int kGrabsAhead = 1;
constexpr int kGrabMax = 4;

template <int DIM, int TESS, bool POW2>
__global__ void __launch_bounds__(1024)
    k_integrate_items(const WorkItem* __restrict__ items, int nItems, int chunk, unsigned int* __restrict__ queue,
                      double h, int nT, int nS, int sort_off, int sort_cap) {
  constexpr int NE = DIM * (DIM + 1);
  extern __shared__ double lds[];
  __shared__ int s_t0, s_t1, cursor, grid_w;
  // sort_off > 0: runs of up to sort_cap points in an order by position (tile_bucket_order)
  unsigned int* hist = reinterpret_cast<unsigned int*>(lds + sort_off);
  uint16_t* idx = reinterpret_cast<uint16_t*>(hist + kBucketMax);
  const double *cur = nullptr, *cur_as = nullptr;  // the tables in LDS (block-uniform)
  int cur_nC = 0;
  for (;;) {
    __syncthreads();
    if (threadIdx.x == 0) {
      const unsigned int seen = __hip_atomic_load(queue, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      const int left = seen < (unsigned int)nItems ? nItems - (int)seen : 0;
      int k = left / (kGrabsAhead * (int)gridDim.x);
      k = k > kGrabMax ? kGrabMax : k;
      k = k < chunk ? chunk : k;
      s_t0 = (int)atomicAdd(queue, (unsigned int)k);
      s_t1 = s_t0 + k;
    }
    __syncthreads();
    const int t0 = s_t0;
    if (t0 >= nItems) break;
    const int t1 = s_t1 < nItems ? s_t1 : nItems;
    for (int t = t0; t < t1;) {
      const WorkItem& it = items[t];
      const int nC = it.nC;
      const double *tr = it.trels, *sa = it.as;
      if (tr != cur || sa != cur_as || nC != cur_nC) {
        __syncthreads();
        for (int i = threadIdx.x; i < nC * NE; i += blockDim.x) {
          lds[i] = tr[i];
          lds[nC * NE + i] = sa[i];
        }
        __syncthreads();
        cur = tr;
        cur_as = sa;
        cur_nC = nC;
      }
      const Geom g = it.g;
      const double* pos0 = it.pos0;
      const int64_t most = sort_off > 0 ? sort_cap : kItemMax;
      int64_t end = it.end;
      for (t++; t < t1; t++) {  // the items that go on where this one ends
        const WorkItem& nx = items[t];
        if (nx.trels != tr || nx.as != sa || nx.pos0 != pos0 || nx.out != it.out || nx.begin != end ||
            nx.g.nC0 != g.nC0 || nx.g.nC1 != g.nC1 || nx.g.nC2 != g.nC2 || nx.g.inc_x != g.inc_x ||
            nx.g.inc_y != g.inc_y || nx.g.inc_z != g.inc_z || nx.end - it.begin > most)
          break;
        end = nx.end;
      }
      for (int64_t at = it.begin; at < end; at += kItemMax) {  // (once, for all but huge items)
        const int n = end - at < kItemMax ? (int)(end - at) : kItemMax;
        const uint16_t* lord = nullptr;
        GridOrder gord;
        RowProbe<DIM> probe;
        if (DIM > 1) probe.load(pos0 + at * DIM, n);
        __syncthreads();  // every wave is done with the previous points
        if (threadIdx.x == 0) {
          cursor = 0;
          grid_w = 0x7fffffff;
        }
        if (sort_off > 0 && n <= sort_cap) {  // (block-uniform)
          tile_bucket_order<DIM>(pos0, at, n, g, hist, idx);
          lord = idx;
        } else {
          __syncthreads();
        }
        if (DIM > 1) {
          probe.vote(n, &grid_w);
          __syncthreads();
          gord = grid_order(grid_w, n);
        }
        integrate_range<DIM, TESS, POW2, 0>(at, n, &cursor, pos0, it.out, lds, lds + nC * NE, h, nT, nS, 0, g,
                                            nullptr, gord, at, lord);
      }
    }
  }
}

}  // namespace cpab
