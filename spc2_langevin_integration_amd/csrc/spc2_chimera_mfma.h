// FP32 chimera pair passes of dense linked cells on the matrix cores, shared by
// the single-system kernels (spc2_pairs.hip) and the batched ones
// (spc2_batch.hip).
//
// The passes need, per particle, sums over the partners within rho of cos phi_j
// and sin phi_j (pass 2: also of a_j cos phi_j, a_j sin phi_j) and their number:
// a 0/1 matrix (16 centres x candidates) times a matrix of partner features.
// Both products run as MFMA:
//  * distances: r^2 - rho^2 of 16 candidates x 16 centres in one
//    v_mfma_f32_16x16x4, (x_j, y_j, |r_j|^2, 1) . (-2 x_i, -2 y_i, 1, |r_i|^2 -
//    rho^2); the sign is the decision;
//  * sums: the decisions as bytes 0 / -1 times the partners' features as signed
//    base-128 digits, v_mfma_i32_16x16x64_i8 over 64 candidates.
// The distance tile's layout (lane: one centre, four candidates) is that of the
// sum's byte operand when its 64 candidates are taken as byte 4 t + r of lane
// group g = candidate 4 g + r of tile t, so that no data crosses lanes between
// the two: the signs are gathered by three byte permutes per four candidates.
//
// Precision.  A feature v in [-1, 1] is rounded from FP64 to a multiple of 2^-27,
// four digits (the FP32 tiles' values were rounded to 2^-25 at 1/2 and above).
// Integer sums are exact, so a particle's sums depend neither on the order nor on
// the grouping of its partners: one rounding per term, where the FP32 partials
// and Kahan sums had one per addition too.  A pair whose r^2 lies within `band` of
// rho^2, wider than the FP32 error of the product form, is decided by the FP64
// reference distance, as in the scalar walks.
//
// A workgroup takes a chunk of 256 slots of a cell row (as pass1_segment), stages
// the three halo rows in LDS, each padded to tiles of 16, and deals the chunk's
// cells to its wavefronts; a cell's centres go 16 to a group, up to three groups
// sharing each tile read.  Tiles at the ends of a cell's runs reach into
// neighbouring cells of the same row: those particles are beyond rho of its
// centres or candidates anyway.  Then a thread per particle finishes it.  A
// workgroup whose halo or centres (a row's last chunk) do not fit, or that holds
// a value that is not finite, takes the scalar walk of visit_integer: the same
// decisions and integer sums.
//
// Against the FP64 form (N = 50,000, density 4000, rms over the particles): phase
// derivative 1.0e-7 -> 3.0e-9 of its rms, additional terms 1.0e-7 -> 3.0e-9 and
// 8.5e-8 -> 1.9e-8.
//
// Bound: per 64 candidates and group 144 cycles of MFMA (4 x 32 + 16) beside 26
// vector instructions; as measured the phases' latencies (tables, staging,
// epilogue) at 4 wavefronts per SIMD keep vector issue at 55%.  The pair kernel of
// the 512-replica sweep's SE step 1019 -> 649 us (N = 1M alone: pass 1 139 us, pass
// 2 160 us).  On the way there: four groups per tile read held 168 registers (3
// wavefronts, 735 us); the chunk's frame for the products instead of the cell's
// needs a band 30 times wider, whose FP64 decisions cost more than the shift.
// Taken from kMfmaPerCell = 20 particles per cell to where the halo fits the LDS
// (configure_segments_kp); in sparser cells more of a group's
// 16 centres are padding.  At N = 200,000, pass 1 and both SRK passes, the scalar
// walk against this: 24 and 71 against 34 and 75 us at 11 per cell, 27 and 81 against
// 34 and 74 at 16, 33 and 96 against 33 and 80 at 24.  (A small system alone would
// gain from 9 on: 20 and 43 against 12 and 27 us at N = 20,000; but the choice is a
// replica's too, whose batch fills the device.)  Compiled with -ffp-contract=off.
#pragma once

#include "spc2_lds_stencil.h"

namespace spc2 {
namespace {

typedef float v4f __attribute__((ext_vector_type(4)));
typedef int v4i __attribute__((ext_vector_type(4)));

constexpr int kMfmaShort = 64;         // slots of a short chunk (configure_segments)
constexpr int kMfmaTile = 16;          // candidates per tile, centres per group
constexpr int kMfmaWindow = kPairBlock;  // centres of a workgroup at most
constexpr float kMfmaFar = 1.0e6f;     // x and y of the padding candidates

// Feature rows of 16 candidates: the four digits of cos, of sin, then ones (pass
// 1) or the digits of a_j cos and a_j sin (pass 2).
template <int PASS>
struct MfmaLds {
  static constexpr int rows = PASS == 1 ? 9 : 16;
  static constexpr int tile_bytes = kMfmaTile * (8 + rows);
  // (lanes of the rows that pass 1 leaves out read up to 112 bytes further, unused)
  static constexpr int tail_bytes = 128 + kMfmaWindow * (PASS == 1 ? 2 * 8 + 4 : 4 * 8);
  static constexpr int bytes(int cap) { return cap / kMfmaTile * tile_bytes + tail_bytes; }
  float2 *xy;     // positions in the chunk's frame
  uint8_t *feat;  // [tile][rows][16]
  long long *sum;  // [2 or 4][kMfmaWindow]
  int *count;      // [kMfmaWindow] (pass 1)
  __device__ __forceinline__ MfmaLds(void *base, int cap) {
    xy = (float2 *)base;
    sum = (long long *)((char *)base + (size_t)cap * 8);
    count = (int *)(sum + (PASS == 1 ? 2 : 4) * kMfmaWindow);
    feat = (uint8_t *)(count + (PASS == 1 ? kMfmaWindow : 0));
  }
};

// What a particle contributes to its partners' sums: two features (cos and sin
// of its phase, or those times a_j / aj) as packed fixed-point numbers
// (pack_fixed), the first two written with its tile, the others by pass 1.
template <int PASS>
struct Fixed {
  uint32_t v[PASS == 1 ? 2 : 4];
  __device__ __forceinline__ Fixed(const float4 &tile, const uint2 *aq, int k) {
    v[0] = __float_as_uint(tile.z);
    v[1] = __float_as_uint(tile.w);
    if constexpr (PASS == 2) {
      const uint2 q = aq[k];
      v[2] = q.x;
      v[3] = q.y;
    }
  }
  __device__ __forceinline__ bool odd() const {
    bool o = (v[0] == kFixedOdd) | (v[1] == kFixedOdd);
    if constexpr (PASS == 2) o |= (v[2] == kFixedOdd) | (v[3] == kFixedOdd);
    return o;
  }
};

// A particle's integer sums over its partners, and their number.
template <int PASS>
struct IntSums {
  long long v[PASS == 1 ? 2 : 4];
  int n;
  bool odd;  // a partner whose features are not finite
};

// A packed feature's value in two byte products, of its two lower and its two upper
// digits (128 as a byte is -128): -(d0 + 128 d1) and -(d2 + 128 d3) added to lo, hi.
// |lo|, |hi| <= 8256 per feature, so that 2^17 of them stay within 32 bits.
struct FixedHalves {
  int lo = 0, hi = 0;
  __device__ __forceinline__ void add(uint32_t v) {
    lo = __builtin_amdgcn_sdot4((int)v, 0x000080ff, lo, false);
    hi = __builtin_amdgcn_sdot4((int)v, (int)0x80ff0000u, hi, false);
  }
  __device__ __forceinline__ long long value() const { return -((long long)hi * 16384 + lo); }
};
constexpr int kHalvesRun = 1 << 17;

// The scalar walk over the global tiles of slot k in cell c, four candidates
// requested at a time, two byte products per feature and no branch but the band's.
// Bound by the latency of its loads.  An SRK step at N = 20,000 in 10 x 10 cells, no
// workgroup staged: 513 us; 1022 with the features unpacked and added in 64 bits
// behind each decision, 738 with the FP32 form's walk (visit_global).
template <int PASS>
__device__ __forceinline__ int visit_integer(const KParams &P, const int *start, const Tiles &t, const uint2 *aq, int c,
                                             int k, IntSums<PASS> &o) {
  constexpr int F = PASS == 1 ? 2 : 4;
  const int cx = c % P.nx, cy = c / P.nx;
  const float4 u = t.f4[k];
  int cand = 0;
  for (int dyo = -1; dyo <= 1; ++dyo) {
    const int row = adjust_cell(cy + dyo, P.ny) * P.nx;
    const float oy = __builtin_fmaf((float)dyo, P.hyf, -u.y);
    for (int dxo = -1; dxo <= 1; ++dxo) {
      const int jc = row + adjust_cell(cx + dxo, P.nx);
      const float ox = __builtin_fmaf((float)dxo, P.hxf, -u.x);
      const int end = start[jc + 1];
      cand += end - start[jc];
      for (int r0 = start[jc]; r0 < end; r0 += kHalvesRun) {
        const int r1 = min(end, r0 + kHalvesRun);
        FixedHalves h[F];
#pragma unroll 1
        for (int m = r0; m < r1; m += 4) {
          float4 v[4];
          uint2 q[4];
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int j = min(m + i, r1 - 1);
            v[i] = t.f4[j];
            if (PASS == 2) q[i] = aq[j];
          }
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float dx = v[i].x + ox, dy = v[i].y + oy;
            const float r2 = __builtin_fmaf(dx, dx, dy * dy);
            bool in = (r2 <= P.rho2f_hi) & (m + i < r1) & (m + i != k);
            if ((r2 >= P.rho2f_lo) & in) in = exact_r2(t.x, t.y, k, m + i, P.Lx, P.r2Lx, P.Ly, P.r2Ly) <= P.rho2;
            const Fixed<PASS> f(v[i], q + i, 0);
            o.odd |= in & f.odd();
#pragma unroll
            for (int w = 0; w < F; ++w) h[w].add(in ? f.v[w] : 0u);
            o.n += in;
          }
        }
#pragma unroll
        for (int w = 0; w < F; ++w) o.v[w] += h[w].value();
      }
    }
  }
  return cand - 1;
}

// min(m, |a|, |b|) of an MFMA's results a, b.  One instruction (the compiler's
// fminf first makes each operand canonical); `after` is a value it formed from
// the same results, so that the wait they need has passed.
__device__ __forceinline__ float min3_abs(float m, float a, float b, uint32_t after) {
  float r;
  asm("v_min3_f32 %0, %1, |%2|, |%3|" : "=v"(r) : "v"(m), "v"(a), "v"(b), "v"(after));
  return r;
}

// The staged halo rows: row r's first cell at LDS candidate base(r), each row
// padded to whole tiles, then a tile of padding (far).
struct MfmaRows {
  int base1, base2, total;    // base of rows 1, 2 (row 0: 0); all candidates
  int cell1, cell2;           // compact offsets (SegShared) of rows 1, 2 (row 0: 0)
  __device__ __forceinline__ int base(int r) const { return r == 0 ? 0 : (r == 1 ? base1 : base2); }
  __device__ __forceinline__ int cell0(int r) const { return r == 0 ? 0 : (r == 1 ? cell1 : cell2); }
  __device__ __forceinline__ int at(int r, int off) const { return off - cell0(r) + base(r); }
};

// Sums of the centres [c0, c1) (LDS candidates, at most 16 NG of them, of halo
// column q) into lds.sum / count at [c0 - w0, c1 - w0).  k_of_w0: the slot of
// candidate w0.
template <int PASS, int NG>
__device__ __forceinline__ void mfma_cell(const KParams &P, const Tiles &t, const SegShared &sh, const Seg &g,
                                          const MfmaRows &rows, const MfmaLds<PASS> &lds, int q, int c0, int c1, int w0,
                                          int k_of_w0, float band) {
  const float x0 = ((float)(q - (g.ncol >> 1)) + 0.5f) * P.hxf;  // the cell's middle in the chunk's frame
  const int lane = threadIdx.x & 63, n = lane & 15, lg = lane >> 4;
  // the tiles of the cell's three runs in turn: lane l holds the l-th of them (the
  // far tile past the last), 64 at a time
  int T0[3], len[3];
#pragma unroll
  for (int r = 0; r < 3; ++r) {
    const int lo = rows.at(r, sh.off[r * g.ncol + q - 1]), hi = rows.at(r, sh.off[r * g.ncol + q + 2]);
    T0[r] = lo >> 4;
    len[r] = hi > lo ? ((hi + 15) >> 4) - T0[r] : 0;
  }
  const int far = rows.total >> 4;
  const int ntiles = __builtin_amdgcn_readfirstlane(len[0] + len[1] + len[2]);
  const auto tile_list = [&](int first) {
    const int i = first + lane;
    return i < len[0] ? T0[0] + i
                      : (i < len[0] + len[1] ? T0[1] + i - len[0]
                                             : (i < ntiles ? T0[2] + i - len[0] - len[1] : far));
  };
  const v4f zero = {0.0f, 0.0f, 0.0f, 0.0f};
  float b[NG];
  v4i acc[NG];
#pragma unroll
  for (int u = 0; u < NG; ++u) {
    const int ci = c0 + 16 * u + n;
    const bool valid = ci < c1;
    const float2 p = lds.xy[valid ? ci : c0];
    const float x = p.x - x0, nn = __builtin_fmaf(x, x, p.y * p.y);
    const float v = lg == 0 ? -2.0f * x : (lg == 1 ? -2.0f * p.y : (lg == 2 ? 1.0f : nn - P.rho2f));
    b[u] = valid ? v : (lg == 3 ? 1.0e12f : 0.0f);
    acc[u] = v4i{0, 0, 0, 0};
  }
  const float2 *pa = lds.xy + n;
  const uint8_t *pf = lds.feat + n * kMfmaTile + 4 * lg;
  constexpr int kFeat = MfmaLds<PASS>::rows * kMfmaTile;
  int list = tile_list(0);
  int tt[4];
  float2 an[4];
  v4i fn;
  // requests four tiles: the list's i-th and the three after it
  const auto request = [&](int i) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      tt[j] = __builtin_amdgcn_readlane(list, (i & 63) + j);
      an[j] = pa[tt[j] * kMfmaTile];
      fn[j] = *(const int *)(pf + tt[j] * kFeat);
    }
  };
  request(0);
#pragma unroll 1
  for (int i = 0; i < ntiles; i += 4) {
    const int t0 = tt[0], t1 = tt[1], t2 = tt[2], t3 = tt[3];
    const v4i f = fn;
    float a[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float x = an[j].x - x0, y = an[j].y, nn = __builtin_fmaf(x, x, y * y);
      a[j] = lg == 0 ? x : (lg == 1 ? y : (lg == 2 ? nn : 1.0f));
    }
    if (i + 4 < ntiles) {  // the next four, requested before these are used
      if (((i + 4) & 63) == 0) list = tile_list(i + 4);
      request(i + 4);
    }
    v4i m[NG];
    float near[NG];
#pragma unroll
    for (int u = 0; u < NG; ++u) near[u] = 1.0e12f;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      __builtin_amdgcn_sched_barrier(0);  // a tile's distances at a time (registers)
      v4f d[NG];
#pragma unroll
      for (int u = 0; u < NG; ++u) d[u] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[j], b[u], zero, 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int u = 0; u < NG; ++u) {
        // byte k = the sign of d[k]: 0xff within rho
        const uint32_t lo = __builtin_amdgcn_perm(__float_as_uint(d[u][1]), __float_as_uint(d[u][0]), 0x0c0c0b09u);
        const uint32_t hi = __builtin_amdgcn_perm(__float_as_uint(d[u][3]), __float_as_uint(d[u][2]), 0x0b090c0cu);
        m[u][j] = (int)(lo | hi);
        near[u] = min3_abs(min3_abs(near[u], d[u][0], d[u][1], lo), d[u][2], d[u][3], hi);
      }
    }
#pragma unroll
    for (int u = 0; u < NG; ++u) {
      // some pair in the band: the distances again, and the FP64 decision for it
      if (__builtin_expect(__any(near[u] <= band), 0)) {
        uint32_t todo = 0, in = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          __builtin_amdgcn_sched_barrier(0);
          const v4f d = __builtin_amdgcn_mfma_f32_16x16x4f32(a[j], b[u], zero, 0, 0, 0);
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            todo |= __builtin_fabsf(d[k]) <= band ? 1u << (4 * j + k) : 0u;
            in |= d[k] < 0.0f ? 1u << (4 * j + k) : 0u;
          }
        }
        while (todo) {
          const int bit = __builtin_ctz(todo), j = bit >> 2;
          todo &= todo - 1u;
          const int cj = 16 * (j == 0 ? t0 : (j == 1 ? t1 : (j == 2 ? t2 : t3))) + 4 * lg + (bit & 3);
          const int rr = cj >= rows.base2 ? 2 : (cj >= rows.base1 ? 1 : 0);
          const int el = cj - rows.base(rr) + rows.cell0(rr);
          const int s = find_slot(sh, g.ns, el);
          const int kj = sh.gst[s] + (el - sh.off[s]), ki = k_of_w0 + (c0 + 16 * u + n - w0);
          const bool near_in = exact_r2(t.x, t.y, ki, kj, P.Lx, P.r2Lx, P.Ly, P.r2Ly) <= P.rho2;
          in = near_in ? in | 1u << bit : in & ~(1u << bit);
        }
#pragma unroll
        for (int j = 0; j < 4; ++j)  // four bits to four bytes 0 / 0xff
          m[u][j] = (int)((((in >> (4 * j)) & 15u) * 0x00204081u & 0x01010101u) * 0xffu);
      }
    }
#pragma unroll
    for (int u = 0; u < NG; ++u) acc[u] = __builtin_amdgcn_mfma_i32_16x16x64_i8(f, m[u], acc[u], 0, 0, 0);
  }
  // lane (n, lg) holds feature lg of centre n: its digits, times -1
#pragma unroll
  for (int u = 0; u < NG; ++u) {
    const int ci = c0 + 16 * u + n;
    if (ci >= c1) continue;
    const long long v = -((((long long)acc[u][3] * 128 + acc[u][2]) * 128 + acc[u][1]) * 128 + acc[u][0]);
    if (PASS == 2 || lg < 2) lds.sum[lg * kMfmaWindow + (ci - w0)] = v;
    if (PASS == 1 && lg == 2) lds.count[ci - w0] = -acc[u][0];
  }
}

// One pair workgroup: pass1_segment / pass2_segment of a dense FP32 chimera system.
// SHORT: for chunks of at most kMfmaShort slots, of fewer cells than wavefronts,
// whose groups of centres then go to a wavefront each (an instance of its own: in
// one kernel the two walks' registers cost a batch's pass 13%).
template <int PASS, int EPI, bool SHORT>
__device__ __forceinline__ void mfma_segment(const KParams &P, const int *__restrict__ start, const Tiles &t,
                                             const int *__restrict__ slot_h, const int *__restrict__ slot_id,
                                             const double *gp, const EpiCtx &e, unsigned long long *counts, int seg,
                                             SegShared &sh, void *dyn_lds) {
  Block b;
  if (!block_range(P, start, t, seg, b)) return;  // the whole workgroup
  const bool fits = b.W <= kMaxSegW;
  Seg g{};
  MfmaRows rows{};
  if (fits) {
    g = halo_setup(P, start, b.cy, b.cx0, b.W, sh);
    rows.cell1 = sh.off[g.ncol];
    rows.cell2 = sh.off[2 * g.ncol];
    rows.base1 = (rows.cell1 + 15) & ~15;
    rows.base2 = rows.base1 + ((rows.cell2 - rows.cell1 + 15) & ~15);
    rows.total = rows.base2 + ((g.total - rows.cell2 + 15) & ~15);
  }
  const int ncen = b.k1 - b.k0;
  bool staged = fits && rows.total + kMfmaTile <= P.lds_cap && ncen <= kMfmaWindow;
  const MfmaLds<PASS> lds(dyn_lds, P.lds_cap);
  bool fit = true;
  if (staged) {
    // A halo row's cells are consecutive slots but for the columns that wrap: its
    // first cell alone, the middle ones, its last cell alone.
    const int qc = g.ncol >> 1;  // the chunk's frame: x from the middle column's edge
    const int qa = g.cx0 == 0 ? 1 : 0, qb = g.cx0 + g.W >= P.nx ? g.W + 1 : g.W + 2;
    struct Row {
      int len, ea, eb, s0, s1, s2, cell0;
    } row[3];
#pragma unroll
    for (int r = 0; r < 3; ++r) {
      const int rb = r * g.ncol;
      Row &w = row[r];
      w.len = sh.off[rb + g.ncol] - sh.off[rb];
      w.ea = sh.off[rb + qa] - sh.off[rb];
      w.eb = sh.off[rb + qb] - sh.off[rb];
      // slot of the row's el-th candidate, less el
      w.s0 = sh.gst[rb];
      w.s1 = sh.gst[rb + qa] - w.ea;
      w.s2 = qb < g.ncol ? sh.gst[rb + qb] - w.eb : 0;
      w.cell0 = adjust_cell(g.cy + r - 1, P.ny) * P.nx + g.cx0 - 1;  // less q: the cell of column 0
    }
    // Two candidates of each row per thread and turn, all six requested before any
    // is used: a turn costs one memory latency, and a halo of 256-slot chunks is
    // one turn.
    const int most = max(row[0].len, max(row[1].len, row[2].len));
    for (int e0 = threadIdx.x; e0 < most + kMfmaTile - 1; e0 += 2 * kPairBlock) {
      float4 v[3][2];
      uint2 aq[3][2];
      int cell[3][2];
#pragma unroll
      for (int r = 0; r < 3; ++r)
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const Row &w = row[r];
          const int el = max(0, min(e0 + i * kPairBlock, w.len - 1));
          const int k = w.len > 0 ? el + (el < w.ea ? w.s0 : (el < w.eb ? w.s1 : w.s2)) : 0;
          v[r][i] = t.f4[k];
          cell[r][i] = t.cell[k];
          if (PASS == 2) aq[r][i] = e.aq[k];
        }
#pragma unroll
      for (int r = 0; r < 3; ++r)
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const Row &w = row[r];
          const int el = e0 + i * kPairBlock, c = rows.base(r) + el;
          if (el >= ((w.len + 15) & ~15)) continue;  // (the row's padding too)
          float x = kMfmaFar, y = kMfmaFar;
          if (el < w.len) {
            const Fixed<PASS> fx(v[r][i], &aq[r][i], 0);
            const int q = el < w.ea ? 0 : (el < w.eb ? cell[r][i] - w.cell0 : g.ncol - 1);
            x = __builtin_fmaf((float)(q - qc), P.hxf, v[r][i].x);
            y = __builtin_fmaf((float)r - 1.5f, P.hyf, v[r][i].y);  // from the centre row's middle
            fit &= (__builtin_fabsf(x) < kMfmaFar) & (__builtin_fabsf(y) < kMfmaFar) & !fx.odd();
            uint8_t *fb = lds.feat + (c >> 4) * (MfmaLds<PASS>::rows * kMfmaTile) + (c & 15);
#pragma unroll
            for (int w = 0; w < (PASS == 1 ? 2 : 4); ++w)
#pragma unroll
              for (int k = 0; k < 4; ++k) fb[(4 * w + k) * kMfmaTile] = (uint8_t)(fx.v[w] >> (8 * k));
            if (PASS == 1) fb[8 * kMfmaTile] = 1;
          }
          lds.xy[c] = make_float2(x, y);
        }
    }
    if (threadIdx.x < kMfmaTile) lds.xy[rows.total + threadIdx.x] = make_float2(kMfmaFar, kMfmaFar);  // the far tile
  }
  staged = __syncthreads_and(staged && fit);
  // FP32 error of r^2: the product form's in a cell's own frame (|x|, |y| <= 1.5
  // cells: below 2e-6 of a cell squared) and the staged coordinates' (2^-24 of the
  // chunk's half width each, times 2 rho)
  const float band = P.band_rho2f + 3.0e-7f * P.rhof * (0.5f * (float)b.W + 2.0f) * P.hxf;
  const int c0 = staged ? rows.at(1, sh.off[g.ncol + 1] + (b.k0 - sh.gst[g.ncol + 1])) : 0;  // candidate of slot k0
  long long cand_sum = 0, n_sum = 0;
  if (staged) {
    const int wave = threadIdx.x >> 6, c1 = c0 + ncen;
    int unit = 0;
    if (SHORT) {
      for (int q = 1; q <= g.W; ++q) {
        int a = __builtin_amdgcn_readfirstlane(max(c0, rows.at(1, sh.off[g.ncol + q])));
        const int z = __builtin_amdgcn_readfirstlane(min(c1, rows.at(1, sh.off[g.ncol + q + 1])));
        for (; a < z; a += 16, ++unit)
          if ((unit & 3) == wave) mfma_cell<PASS, 1>(P, t, sh, g, rows, lds, q, a, min(z, a + 16), c0, b.k0, band);
      }
    } else {
      for (int q = 1; q <= g.W; ++q) {
        int a = __builtin_amdgcn_readfirstlane(max(c0, rows.at(1, sh.off[g.ncol + q])));
        const int z = __builtin_amdgcn_readfirstlane(min(c1, rows.at(1, sh.off[g.ncol + q + 1])));
        if (a >= z || (unit++ & 3) != wave) continue;
        while (a < z) {  // at most three groups at a time (registers), four as two and two
          const int left = (z - a + 15) >> 4, groups = left == 4 ? 2 : min(3, left), ce = min(z, a + 16 * groups);
          if (groups == 3) mfma_cell<PASS, 3>(P, t, sh, g, rows, lds, q, a, ce, c0, b.k0, band);
          else if (groups == 2) mfma_cell<PASS, 2>(P, t, sh, g, rows, lds, q, a, ce, c0, b.k0, band);
          else mfma_cell<PASS, 1>(P, t, sh, g, rows, lds, q, a, ce, c0, b.k0, band);
          a = ce;
        }
      }
    }
    __syncthreads();
  }
  // (a loop of its own: around the walk too, the compiler would keep the
  // epilogue's constants in registers through the walk)
  for (int p = threadIdx.x; p < ncen; p += kPairBlock) {
    {
      const int k = b.k0 + p, h = slot_h[k], id = slot_id[k];
      IntSums<PASS> o{};
      int cand = 0;
      if (staged) {
        const Fixed<PASS> own(t.f4[k], e.aq, k);
#pragma unroll
        for (int q = 0; q < (PASS == 1 ? 2 : 4); ++q)  // less the particle itself
          o.v[q] = lds.sum[q * kMfmaWindow + p] - unpack_fixed(own.v[q]);
        if (PASS == 1) o.n = lds.count[p] - 1;
        if (counts) {
          const int q = t.cell[k] - b.cy * P.nx - g.cx0 + 1;
          for (int r = 0; r < 3; ++r) cand += sh.off[r * g.ncol + q + 2] - sh.off[r * g.ncol + q - 1];
          --cand;
        }
      } else {
        cand = visit_integer<PASS>(P, start, t, e.aq, t.cell[k], k, o);
      }
      const double nan = __builtin_nan("");
      const double phase = gp[h];
      double sa, ca;
      sincos(phase + P.alpha, &sa, &ca);
      const double C = o.odd ? nan : (double)o.v[0] * kFixedUnit;
      const double S = o.odd ? nan : (double)o.v[1] * kFixedUnit;
      if constexpr (PASS == 1) {
        Pass1Out r{};
        const double A = ca * S - sa * C;
        r.phase = phase;
        r.n = o.n;
        r.written = r.n != 0;
        r.aphi = r.n != 0 ? P.sigma * A / (double)r.n : 0.0;
        const EpiState st = epilogue1<EPI>(P, e, h, id, k, r);
        bin_stage<EPI>(P, e, h, id, st);
        if constexpr (EPI == EPI_ITO1) {  // pass 2's features
          const double a = st.ap * P.raj;
          const Fixed<1> own(t.f4[k], nullptr, k);
          const double c = (double)unpack_fixed(own.v[0]) * kFixedUnit, s = (double)unpack_fixed(own.v[1]) * kFixedUnit;
          const bool ok = !own.odd() & (__builtin_fabs(a) <= 1.0);
          e.aq[k] = ok ? make_uint2(pack_fixed(a * c), pack_fixed(a * s)) : make_uint2(kFixedOdd, kFixedOdd);
        }
        cand_sum += cand;
        n_sum += r.n;
      } else {
        const double aj = P.aj * kFixedUnit;
        const double Pc = o.odd ? nan : (double)o.v[2] * aj, Qs = o.odd ? nan : (double)o.v[3] * aj;
        const double ai = e.aphi_slot[k], n = e.n_slot[k];
        double a0 = EPI == EPI_ITO2 ? e.a0[h] : 0.0, a1 = EPI == EPI_ITO2 ? e.a1[h] : 0.0;
        if (n != 0) {
          const double sc = ca * C + sa * S;
          a0 += sc / n;
          a1 += (ca * Pc + sa * Qs - ai * sc) / n;
        }
        Pass2Out r;
        r.phase = phase;
        r.ai = ai;
        r.a0 = a0 * -sqrt(2.0 * P.D);
        r.a1 = a1 + -2.0 * P.D * ai;
        epilogue2<EPI>(P, e, h, id, r);
      }
    }
  }
  if (counts) count_add(counts, cand_sum, n_sum, 0);
}

}  // namespace
}  // namespace spc2
