// Linked-cell build on gfx950: stage + binning (histogram and per-cell lists, also
// done by a pass's epilogue for the next build), a wavefront scan of the histogram,
// and a stable counting sort that writes the cell-sorted tiles the pair kernels
// read.  Compiled with -ffp-contract=off.
//
// Particle data live in "home" order h (a permutation of the particle ids kept
// close to cell order, see spc2_api.hip); hid[h] is the particle id at home h.
// The cell list itself is the reference's: cells in row-major order, members
// in ascending particle id.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "spc2_device.h"
#include "spc2_internal.h"

namespace spc2 {

namespace {

constexpr int kBlock = 256;
constexpr int kScanItems = 4;                   // counts per thread
constexpr int kScanTile = kBlock * kScanItems;  // counts per workgroup

inline int blocks_for(long long n, int b = kBlock) { return (int)((n + b - 1) / b); }

// K1: stage s + (k_coef * dt) * k (ChimeraSystem.cpp:274-276, evaluated as
// (k_coef * dt) * k_prev like the reference); on the linked-cell path the
// position is wrapped if outside the box and binned (ChimeraSystem.cpp:291-309).
// apf4 (the FP32 form on the all-pairs path): each particle's tile, whose cos and
// sin of the stage phase the pair sums read instead of an FP64 sincos per pair (the
// same values).
__global__ __launch_bounds__(kBlock) void k_stage_bin(int n, int linked, Box b, int nx, int ny, const double *sx,
                                                      const double *sy, const double *sp, const double *kx,
                                                      const double *ky, const double *kp, double kcdt, double *gx,
                                                      double *gy, double *gp, const int *hid, Bins bins, int cap,
                                                      float4 *apf4) {
  const int h = blockIdx.x * blockDim.x + threadIdx.x;
  const bool valid = h < n;
  int c = 0;
  if (valid) {
    double x = sx[h], y = sy[h], p = sp[h];
    if (kx) {
      x = x + kcdt * kx[h];
      y = y + kcdt * ky[h];
      p = p + kcdt * kp[h];
    }
    if (linked) {
      cond_wrap(b, x, y);
      c = cell_coord(y, b.Ly, ny) * nx + cell_coord(x, b.Lx, nx);
      bins.cell_of[h] = c;
    }
    gx[h] = x;
    gy[h] = y;
    gp[h] = p;
    if (apf4) {
      double sn, cs;
      sincos(p, &sn, &cs);
      apf4[h] = make_float4((float)x, (float)y, (float)cs, (float)sn);
    }
  }
  if (linked) bin_particle(bins, c, cap, h, valid && cap ? hid[h] : 0, valid);
}

// Inclusive scan of one int per thread across a 256-thread workgroup:
// shuffles inside each 64-lane wavefront, wavefront totals through LDS.
__device__ __forceinline__ int block_inclusive_scan(int v, int *wtot) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    int u = __shfl_up(v, d, 64);
    if (lane >= d) v += u;
  }
  if (lane == 63) wtot[w] = v;
  __syncthreads();
  int add = 0;
#pragma unroll
  for (int q = 0; q < kBlock / 64; ++q) add += (q < w) ? wtot[q] : 0;
  __syncthreads();
  return v + add;
}

// K2a: per-workgroup totals of kScanTile consecutive counts.
__global__ __launch_bounds__(kBlock) void k_scan_reduce(const int *count, int nc, int *bsum) {
  __shared__ int wtot[kBlock / 64];
  const int base = blockIdx.x * kScanTile + threadIdx.x * kScanItems;
  int s = 0;
#pragma unroll
  for (int q = 0; q < kScanItems; ++q) s += (base + q < nc) ? count[base + q] : 0;
  int incl = block_inclusive_scan(s, wtot);
  if (threadIdx.x == kBlock - 1) bsum[blockIdx.x] = incl;
}

// K2b: exclusive scan of the workgroup totals (one workgroup, carried tiles);
// writes the grand total to start[nc].
__global__ __launch_bounds__(kBlock) void k_scan_bsum(int *bsum, int nb, int *start, int nc) {
  __shared__ int wtot[kBlock / 64];
  __shared__ int carry;
  if (threadIdx.x == 0) carry = 0;
  __syncthreads();
  for (int base = 0; base < nb; base += kBlock) {
    int i = base + threadIdx.x;
    int v = i < nb ? bsum[i] : 0;
    int incl = block_inclusive_scan(v, wtot);
    int c0 = carry;
    if (i < nb) bsum[i] = c0 + incl - v;
    __syncthreads();
    if (threadIdx.x == kBlock - 1) carry = c0 + incl;
    __syncthreads();
  }
  if (threadIdx.x == 0) start[nc] = carry;
}

// K2c: exclusive scan inside each tile plus the tile offset -> start[];
// clears the histogram for the next build.
__global__ __launch_bounds__(kBlock) void k_scan_apply(int *count, int nc, const int *bsum, int *start) {
  __shared__ int wtot[kBlock / 64];
  const int base = blockIdx.x * kScanTile + threadIdx.x * kScanItems;
  int v[kScanItems];
  int s = 0;
#pragma unroll
  for (int q = 0; q < kScanItems; ++q) {
    v[q] = (base + q < nc) ? count[base + q] : 0;
    s += v[q];
  }
  int run = block_inclusive_scan(s, wtot) - s + bsum[blockIdx.x];
#pragma unroll
  for (int q = 0; q < kScanItems; ++q) {
    if (base + q < nc) {
      start[base + q] = run;
      count[base + q] = 0;
    }
    run += v[q];
  }
}

// K2 for at most kScanSingle counts: the whole exclusive scan in one
// workgroup, tile by tile with a carried total (the three-launch scan's values),
// writing start[nc] and clearing the histogram.
constexpr int kScanSingle = 4 * kScanTile;
__global__ __launch_bounds__(kBlock) void k_scan_single(int *count, int nc, int *start) {
  __shared__ int wtot[kBlock / 64];
  __shared__ int carry;
  if (threadIdx.x == 0) carry = 0;
  __syncthreads();
  for (int tile = 0; tile < nc; tile += kScanTile) {
    const int base = tile + threadIdx.x * kScanItems;
    int v[kScanItems];
    int s = 0;
#pragma unroll
    for (int q = 0; q < kScanItems; ++q) {
      v[q] = (base + q < nc) ? count[base + q] : 0;
      s += v[q];
    }
    int run = carry + block_inclusive_scan(s, wtot) - s;
#pragma unroll
    for (int q = 0; q < kScanItems; ++q) {
      if (base + q < nc) {
        start[base + q] = run;
        count[base + q] = 0;
      }
      run += v[q];
    }
    __syncthreads();  // every lane has read carry
    if (threadIdx.x == kBlock - 1) carry = run;
    __syncthreads();
  }
  if (threadIdx.x == 0) start[nc] = carry;
}

// Counts summed together by k_sort_tiles, and how many such sums it takes.
constexpr int kBinRow = 16;
constexpr int kMaxBinRows = 4 * kBlock;

// The particle of home h, cell c and id in the cell-sorted slot dst.
template <int PREC>
__device__ __forceinline__ void write_slot(int dst, int h, int id, int c, int nx, int fixed, double hx, double hy,
                                           const double *gx, const double *gy, const double *gp, int *slot_h,
                                           int *slot_id, const Tiles &t) {
  slot_h[dst] = h;
  slot_id[dst] = id;
  t.cell[dst] = c;
  double x = gx[h], y = gy[h], p = gp[h];
  if (PREC == P32K) {
    int cx = c % nx, cy = c / nx;
    double sn, cs;
    sincos(p, &sn, &cs);
    // fixed: cos and sin as the matrix-core passes' packed features
    t.f4[dst] = make_float4((float)(x - (double)cx * hx), (float)(y - (double)cy * hy),
                            fixed ? __uint_as_float(pack_fixed(cs)) : (float)cs,
                            fixed ? __uint_as_float(pack_fixed(sn)) : (float)sn);
    t.x[dst] = x;
    t.y[dst] = y;
  } else {
    t.x[dst] = x;
    t.y[dst] = y;
    t.p[dst] = p;
    if (PREC == P64F) {
      double sn, cs;
      sincos(p, &sn, &cs);
      t.c[dst] = cs;
      t.s[dst] = sn;
    }
  }
}

// K3a: place each particle at cell start + arrival rank (home and id).
__global__ __launch_bounds__(kBlock) void k_place(int n, const int *cell_of, const int *local, const int *start,
                                                  const int *hid, int *tmp, int *tmpid) {
  int h = blockIdx.x * blockDim.x + threadIdx.x;
  if (h >= n) return;
  int pos = start[cell_of[h]] + local[h];
  tmp[pos] = h;
  tmpid[pos] = hid[h];
}

// K3b: stable counting sort.  The final position of a particle inside its cell
// is the number of cell members with a smaller particle id, which reproduces
// the reference's ascending push_back order (ChimeraSystem.cpp:335-338).  The
// same thread gathers the particle's stage data into the cell-sorted tiles.
template <int PREC>
__global__ __launch_bounds__(kBlock) void k_rank_tiles(int n, int nx, int fixed, double hx, double hy, const int *tmp,
                                                       const int *tmpid, const int *cell_of, const int *start,
                                                       const double *gx, const double *gy, const double *gp,
                                                       int *slot_h, int *slot_id, Tiles t) {
  __shared__ int ids[kRankStage];
  __shared__ int span[2];
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  int h = 0, id = 0, c = 0, lo = 0, hi = 0;
  if (k < n) {
    h = tmp[k];
    id = tmpid[k];
    c = cell_of[h];
    lo = start[c];
    hi = start[c + 1];
  }
  const int s0 = stage_cell_ids(ids, span, tmpid, n, lo, hi);
  if (k >= n) return;
  const int r = s0 >= 0 ? rank_in_cell(ids + (lo - s0), hi - lo, id) : rank_in_cell(tmpid + lo, hi - lo, id);
  const int dst = lo + r;
  write_slot<PREC>(dst, h, id, c, nx, fixed, hx, hy, gx, gy, gp, slot_h, slot_id, t);
}

// K2 and K3 in one launch, for the lists of smaller grids: every workgroup sums the
// histogram by kBinRow counts and scans those sums in LDS (they share the writing of
// start[]), then a thread per home finds its cell's start and ranks its id in the
// cell's list.  Reads one set of counts and chains and clears the other, which the
// next binning fills.  Bound by launch and load latencies: 4.2 us at N = 1000 where
// scan, placing and sort take 13.1, 5.8 (13.1) at N = 8191, 5.9 (23.6) at N = 50,000
// and 4900 cells, 23 (32) at N = 600,000 and 15,000 cells.  (With the whole histogram
// scanned in LDS instead, two serial runs over it per thread: 35 us at 14,000 cells.)
template <int PREC>
__global__ __launch_bounds__(kBlock) void k_sort_tiles(int n, int nx, int nc, int fixed, int cap, double hx, double hy,
                                                       Bins bins, int *other, int *other_used, const int *hid, int *start,
                                                       const double *gx, const double *gy, const double *gp,
                                                       int *slot_h, int *slot_id, Tiles t) {
  __shared__ int pre[kMaxBinRows];  // the rows' starts
  __shared__ int wtot[kBlock / 64];
  const int h = blockIdx.x * kBlock + threadIdx.x, all = gridDim.x * kBlock;
  const int rows = (nc + kBinRow - 1) / kBinRow;
  const int4 *count = (const int4 *)bins.count;
  for (int q = h; q < 2 * kBinRow / 4 * rows; q += all) ((int4 *)other)[q] = make_int4(0, 0, 0, 0);
  if (h == 0) *other_used = 0;
  constexpr int kPer = kMaxBinRows / kBlock;
  int own[kPer], sum = 0;
#pragma unroll
  for (int u = 0; u < kPer; ++u) {
    const int q = (int)threadIdx.x + u * kBlock;
    int v = 0;
    if (q < rows) {
#pragma unroll
      for (int w = 0; w < kBinRow / 4; ++w) {
        const int4 c = count[q * (kBinRow / 4) + w];
        v += (c.x + c.y) + (c.z + c.w);
      }
    }
    pre[q] = v;
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < kPer; ++u) {
    own[u] = pre[(int)threadIdx.x * kPer + u];
    sum += own[u];
  }
  int run = block_inclusive_scan(sum, wtot) - sum;
#pragma unroll
  for (int u = 0; u < kPer; ++u) {
    pre[(int)threadIdx.x * kPer + u] = run;
    run += own[u];
  }
  __syncthreads();
  for (int q = h; q < rows; q += all) {
    int at = pre[q];
#pragma unroll
    for (int w = 0; w < kBinRow / 4; ++w) {
      const int4 c = count[q * (kBinRow / 4) + w];
      ((int4 *)start)[q * (kBinRow / 4) + w] = make_int4(at, at + c.x, at + c.x + c.y, at + c.x + c.y + c.z);
      at += (c.x + c.y) + (c.z + c.w);
    }
  }
  if (h == 0 && nc % kBinRow == 0) start[nc] = n;
  if (h >= n) return;
  const int c = bins.cell_of[h], id = hid[h], in_row = c % kBinRow;
  int lo = pre[c / kBinRow];
#pragma unroll
  for (int w = 0; w < kBinRow / 4; ++w) {
    const int4 v = count[c / kBinRow * (kBinRow / 4) + w];
    lo += 4 * w < in_row ? v.x : 0;
    lo += 4 * w + 1 < in_row ? v.y : 0;
    lo += 4 * w + 2 < in_row ? v.z : 0;
    lo += 4 * w + 3 < in_row ? v.w : 0;
  }
  const int dst = lo + rank_in_bin(bins, c, cap, bins.count[c], id);
  write_slot<PREC>(dst, h, id, c, nx, fixed, hx, hy, gx, gy, gp, slot_h, slot_id, t);
}

}  // namespace

void launch_stage_bin(Sim &s, const double *kx, const double *ky, const double *kp, double kcdt) {
  Box b{s.kp.Lx, s.kp.Ly, s.kp.rLx, s.kp.rLy};
  hipLaunchKernelGGL(k_stage_bin, dim3(blocks_for(s.n)), dim3(kBlock), 0, s.stream, s.n, (int)s.linked, b, s.nx,
                     s.ny, s.sx, s.sy, s.sp, kx, ky, kp, kcdt, s.gx, s.gy, s.gp, s.hid, s.bins(), s.kp.bin_cap,
                     !s.linked && s.prec == P32K ? s.t.f4 : nullptr);
}

int scan_blocks(int nc) { return (nc + kScanTile - 1) / kScanTile; }

// Exclusive scan of count[0..m) into out[0..m], out[m] = total; clears count.
// bsum holds scan_blocks(m) + 1 ints.
void launch_scan_raw(hipStream_t st, int *bsum, int *count, int m, int *out) {
  if (m <= kScanSingle) {  // small grids: one launch instead of three
    hipLaunchKernelGGL(k_scan_single, dim3(1), dim3(kBlock), 0, st, count, m, out);
    return;
  }
  const int nb = scan_blocks(m);
  hipLaunchKernelGGL(k_scan_reduce, dim3(nb), dim3(kBlock), 0, st, count, m, bsum);
  hipLaunchKernelGGL(k_scan_bsum, dim3(1), dim3(kBlock), 0, st, bsum, nb, out, m);
  hipLaunchKernelGGL(k_scan_apply, dim3(nb), dim3(kBlock), 0, st, count, m, bsum, out);
}

void launch_scan_array(Sim &s, int *count, int m, int *out) { launch_scan_raw(s.stream, s.bsum, count, m, out); }

void launch_place_raw(hipStream_t st, int n, const int *cell_of, const int *local, const int *start, const int *hid,
                      int *tmp, int *tmpid) {
  hipLaunchKernelGGL(k_place, dim3(blocks_for(n)), dim3(kBlock), 0, st, n, cell_of, local, start, hid, tmp, tmpid);
}

namespace {
template <int PREC>
void launch_sort(Sim &s, const Bins &b) {
  const dim3 g(blocks_for(s.n)), blk(kBlock);
  if (s.kp.bin_cap)
    hipLaunchKernelGGL(k_sort_tiles<PREC>, g, blk, 0, s.stream, s.n, s.nx, s.nc,
                       s.kp.mfma, s.kp.bin_cap, s.kp.hx, s.kp.hy, b, s.bins().count, s.bins().used, s.hid, s.start, s.gx, s.gy, s.gp,
                       s.slot_h, s.slot_id, s.t);
  else
    hipLaunchKernelGGL(k_rank_tiles<PREC>, g, blk, 0, s.stream, s.n, s.nx, s.kp.mfma, s.kp.hx, s.kp.hy, s.tmp, s.tmpid,
                       s.cell_of, s.start, s.gx, s.gy, s.gp, s.slot_h, s.slot_id, s.t);
}
}  // namespace

// Cell starts, order and tiles of the particles binned last.
void launch_cells(Sim &s) {
  const Bins b = s.bins();
  if (s.kp.bin_cap) {
    s.bin_set ^= 1;
  } else {
    launch_scan_array(s, s.count, s.nc, s.start);
    launch_place_raw(s.stream, s.n, s.cell_of, s.local, s.start, s.hid, s.tmp, s.tmpid);
  }
  switch (s.prec) {
    case P64: launch_sort<P64>(s, b); break;
    case P64F: launch_sort<P64F>(s, b); break;
    default: launch_sort<P32K>(s, b);
  }
}

// Lists for cell grids whose histogram every workgroup of the sort can sum by
// itself (16,384 counts, at the most 64 KB read by each); not for Verlet builds, which are rare, find the
// particles far from cell order and then write scattered where k_rank_tiles reads
// scattered (3.86M particles in random order: 470 against 240 us with the placing).
// A list holds its cell's mean and four standard deviations of a uniform state.
void configure_bins(Sim &s) {
  s.kp.bin_cap = 0;
  s.count_stride = std::max(s.nc, 1);
  if (!s.linked || s.verlet || s.nc > kBinRow * kMaxBinRows || s.n >= (1 << 29)) return;  // (3 n ints of chains)
  s.count_stride = (s.nc + kBinRow - 1) / kBinRow * kBinRow;
  const double per_cell = (double)s.n / (double)s.nc;
  s.kp.bin_cap = (int)std::ceil((per_cell + 4.0 * std::sqrt(per_cell) + 8.0) / 4.0) * 4;
}

}  // namespace spc2
