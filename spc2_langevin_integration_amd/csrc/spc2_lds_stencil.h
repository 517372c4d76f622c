// LDS staging of the 3 x 3 cell stencil and the pass-1 / pass-2 bodies of one
// pair workgroup, shared by the single-system kernels (spc2_pairs.hip) and the
// batched kernels (spc2_batch.hip).
//
// Work decomposition: one 256-lane workgroup per row chunk (a run of
// consecutive slots of one cell row, which spans W cells) or, in sparse
// systems, per row segment of W cells.  It stages the 3 x (W + 2) halo cells'
// tiles in LDS with coalesced reads (cells of a row are contiguous in the
// cell-sorted arrays), then each lane takes one centre particle, or in the FP64 forms
// its share of one's candidates.  In LDS the three stencil cells of one stencil row
// are adjacent, so a particle's 9 cells are 3 contiguous ranges, in the reference
// order (cells (-1,dy), (0,dy), (1,dy), ascending particle index inside a cell); a
// lane takes a run of each in that order.  A workgroup whose halo does not fit the LDS
// capacity falls back to reading the same tiles from global memory with the same
// arithmetic and order.  Compiled with -ffp-contract=off.
#pragma once

#include <type_traits>

#include "spc2_pair_accumulators.h"

namespace spc2 {
namespace {

constexpr int kMaxSegW = 64;  // 3 (kMaxSegW + 2) halo cells, one per lane of the setup scan
constexpr int kMaxSlots = 3 * (kMaxSegW + 2);
constexpr double kChunkPerCell = 8.0;  // mean particles per cell from which rows are cut into chunks
// x offset that puts a candidate beyond every cutoff (r^2 about 1e12)
constexpr float kSelfOff = 1.0e6f;


// =============================================================================
// Row-segment setup and LDS staging
// =============================================================================

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
  for (int q = 0; q < kPairBlock / 64; ++q) add += (q < w) ? wtot[q] : 0;
  __syncthreads();
  return v + add;
}

struct SegShared {
  int off[kMaxSlots + 1];  // LDS offset of halo cell (r, q), flattened r * (W + 2) + q; off[3(W+2)] = total
  int gst[kMaxSlots];      // its first global slot
  int wtot[kPairBlock / 64];
};

struct Seg {
  int cy, cx0, W, ncol, ns, total;
};

// Stages the halo table of centre columns cx0 .. cx0 + W - 1 of row cy (W <=
// kMaxSegW): the 3 x (W + 2) cells' first slots and LDS offsets.
__device__ __forceinline__ Seg halo_setup(const KParams &P, const int *start, int cy, int cx0, int W, SegShared &sh) {
  Seg g;
  g.cy = cy;
  g.cx0 = cx0;
  g.W = W;
  g.ncol = g.W + 2;
  g.ns = 3 * g.ncol;
  int cnt = 0;
  if ((int)threadIdx.x < g.ns) {
    int r = threadIdx.x / g.ncol, q = threadIdx.x - r * g.ncol;
    int cyr = adjust_cell(g.cy + r - 1, P.ny);
    int cxq = g.cx0 - 1 + q;
    if (cxq < 0) cxq += P.nx;
    else if (cxq >= P.nx) cxq -= P.nx;
    int cell = cyr * P.nx + cxq;
    int g0 = start[cell];
    cnt = start[cell + 1] - g0;
    sh.gst[threadIdx.x] = g0;
  }
  int incl = block_inclusive_scan(cnt, sh.wtot);
  if ((int)threadIdx.x < g.ns) sh.off[threadIdx.x] = incl - cnt;
  if ((int)threadIdx.x == g.ns - 1) sh.off[g.ns] = incl;
  __syncthreads();
  g.total = sh.off[g.ns];
  return g;
}

// The centre slots [k0, k1) of pair workgroup `seg`, their row cy and the
// columns cx0 .. cx0 + W - 1 they occupy.  Row chunks (P.chunk > 0): slots
// j * chunk .. of the row, the row's last workgroup (j = segs - 1) taking the
// rest; false if the chunk starts past the row.  Row segments: seg_w cells.
struct Block {
  int k0, k1, cy, cx0, W;
};
__device__ __forceinline__ bool block_range(const KParams &P, const int *start, const Tiles &t, int seg, Block &b) {
  b.cy = seg / P.segs;
  const int j = seg - b.cy * P.segs, row = b.cy * P.nx;
  if (P.chunk == 0) {
    b.cx0 = j * P.seg_w;
    b.W = min(P.seg_w, P.nx - b.cx0);
    b.k0 = start[row + b.cx0];
    b.k1 = start[row + b.cx0 + b.W];
    return true;
  }
  const int re = start[row + P.nx];
  b.k0 = start[row] + j * P.chunk;
  if (b.k0 >= re) return false;
  b.k1 = j == P.segs - 1 ? re : min(re, b.k0 + P.chunk);
  b.cx0 = t.cell[b.k0] - row;
  b.W = t.cell[b.k1 - 1] - row - b.cx0 + 1;
  return true;
}

// largest halo slot s with off[s] <= e
__device__ __forceinline__ int find_slot(const SegShared &sh, int ns, int e) {
  int lo = 0, hi = ns - 1;
  while (lo < hi) {
    int mid = (lo + hi + 1) >> 1;
    if (sh.off[mid] <= e) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

// LDS element arrays of one precision and pass, carved from dynamic LDS.
template <int PREC, int PASS>
struct LdsTile;

template <int PASS>
struct LdsTile<P32K, PASS> {
  float4 *f4;
  int *slot;
  float *aj;
  static constexpr int bytes = 20 + (PASS == 2 ? 4 : 0);
  __device__ __forceinline__ LdsTile(void *base, int cap) {
    f4 = (float4 *)base;
    slot = (int *)(f4 + cap);
    aj = (float *)(slot + cap);
  }
  __device__ __forceinline__ void load(int e, int g, const Tiles &t, const EpiCtx &ec) {
    f4[e] = t.f4[g];
    slot[e] = g;
    if (PASS == 2) aj[e] = ec.aphi_slot_f[g];
  }
  __device__ __forceinline__ Src32 src() const { return Src32{f4, slot, aj}; }
};

template <int PREC, int PASS>
struct LdsTile {  // P64 / P64F
  double *x, *y, *a, *b, *aj;
  static constexpr int ncomp = (PREC == P64 ? 3 : 4) + (PASS == 2 ? 1 : 0);
  static constexpr int bytes = 8 * ncomp;
  __device__ __forceinline__ LdsTile(void *base, int cap) {
    x = (double *)base;
    y = x + cap;
    a = y + cap;
    b = a + cap;
    aj = (PREC == P64 ? a : b) + cap;
  }
  __device__ __forceinline__ void load(int e, int g, const Tiles &t, const EpiCtx &ec) {
    x[e] = t.x[g];
    y[e] = t.y[g];
    if (PREC == P64) {
      a[e] = t.p[g];
    } else {
      a[e] = t.c[g];
      b[e] = t.s[g];
    }
    if (PASS == 2) aj[e] = ec.aphi_slot[g];
  }
  __device__ __forceinline__ Src64 src() const {
    return PREC == P64 ? Src64{x, y, a, nullptr, nullptr, aj} : Src64{x, y, nullptr, a, b, aj};
  }
};

// global-memory source over the cell-sorted tiles (overflow fallback)
template <int PREC>
__device__ __forceinline__ typename SrcOf<PREC>::type global_src(const Tiles &t, const EpiCtx &e, int pass) {
  if constexpr (PREC == P32K) {
    return Src32{t.f4, nullptr, pass == 2 ? e.aphi_slot_f : nullptr};
  } else {
    return Src64{t.x, t.y, t.p, t.c, t.s, pass == 2 ? e.aphi_slot : nullptr};
  }
}

// Accumulators with a two-candidate step for the FP32 cell walks.
template <class Acc>
struct HasPair2 : std::false_type {};
template <>
struct HasPair2<ChimAcc<P32K>> : std::true_type {};
template <>
struct HasPair2<Chim2Acc<P32K>> : std::true_type {};
template <>
struct HasPair2<VortAcc<P32K>> : std::true_type {};

// The FP32 walk of one stencil cell, LDS indices [a, b), column offset ox, in
// FP32 partials added to the compensated sums after the cell.  SELF: the cell
// holds the particle itself (LDS index self), which is moved kSelfOff away,
// beyond every cutoff, so it adds the +0 terms of any candidate outside rho
// (partials start at +0 and never become -0, so the sums equal those that skip
// it).  One loop over the cell, not two split at the particle: a wavefront's
// lanes split at different places, so two loops would run the cell twice.
template <bool SELF, class Acc>
__device__ __forceinline__ void cell_run(Acc &acc, const Src32 &src, int a, int b, float ox, int self,
                                         const KParams &P) {
  acc.cell_begin();
  if constexpr (HasPair2<Acc>::value) {
    // the pairs walked by tile address, so that the loop keeps one induction
    // variable, each pair's tiles requested a pair ahead; then the odd last
    // candidate.  The read ahead of the last pair stays within the workgroup's
    // LDS allocation (at most two tiles past the staged halo, in the arrays
    // that follow it) and is not used.
    const float4 *t2 = src.f4 + a, *const last = src.f4 + (b - 1), *const own = src.f4 + self;
    if (t2 < last) {
      // the pair at t2 from the tiles ta, tb; whether another pair follows
      auto step = [&](const float4 &ta, const float4 &tb, int m) {
        const float oxa = SELF && t2 == own ? kSelfOff : ox, oxb = SELF && t2 + 1 == own ? kSelfOff : ox;
        if constexpr (std::is_same<Acc, Chim2Acc<P32K>>::value)  // reads aj[m]: the index too
          acc.pair2_x(src, t2, m, ta, tb, oxa, oxb, P);
        else
          acc.pair2_x(src, t2, ta, tb, oxa, oxb, P);
        t2 += 2;
        return t2 < last;
      };
      // two sets of tile registers taken in turn: each pair's tiles are read
      // into the set the previous pair has just used, with no copies
      float4 a0 = t2[0], b0 = t2[1];
      for (int m = a;; m += 4) {
        const float4 a1 = t2[2], b1 = t2[3];
        if (!step(a0, b0, m)) break;
        a0 = t2[2];
        b0 = t2[3];
        if (!step(a1, b1, m + 2)) break;
      }
    }
    if ((b - a) & 1) acc.template pair_x<SUM_GROUP>(src, b - 1, SELF && b - 1 == self ? kSelfOff : ox, P);
    acc.flush_cell();
  } else {
#pragma unroll 2
    for (int m = a; m < b; ++m) acc.template pair_x<SUM_GROUP>(src, m, SELF && m == self ? kSelfOff : ox, P);
    acc.flush();
  }
}

// Visits the candidates of the centre particle at LDS index ei (halo column qi)
// in reference order, the FP32 forms; returns the number of candidates.
template <class Acc>
__device__ __forceinline__ int visit_lds(Acc &acc, const Src32 &src, const SegShared &sh, int ncol, int qi, int ei,
                                         const KParams &P) {
  int cand = 0;
  // one loop per stencil cell, its column offset computed once (the value the
  // per-candidate selection gives inside that cell), its terms summed in FP32
  // partials that are added to the compensated sums after the cell
#pragma unroll
  for (int r = 0; r < 3; ++r) {
    const int base = r * ncol + qi;
    const int lo = sh.off[base - 1], b1 = sh.off[base], b2 = sh.off[base + 1], hi = sh.off[base + 2];
    acc.row(r - 1, b1, b2, P);
    cand += hi - lo;
    const float ol = acc.co.col(-1), oc = acc.co.col(0), orr = acc.co.col(1);
    cell_run<false>(acc, src, lo, b1, ol, ei, P);
    if (r == 1) cell_run<true>(acc, src, b1, b2, oc, ei, P);
    else cell_run<false>(acc, src, b1, b2, oc, ei, P);
    cell_run<false>(acc, src, b2, hi, orr, ei, P);
  }
  return cand - 1;
}

// The FP64 forms: lane g of the particle's P.lanes lanes takes the g-th of
// P.lanes equal runs of each stencil row's candidates.  The factored form sums a
// candidate where it meets it.  The plain form's terms (a sine or cosine and
// more, 20 to 90 instructions) would run at nearly every candidate if they stood
// behind the distance test, since some lane of the wavefront has a partner there
// although only a third of the candidates are partners.  So the lane first tests
// its candidates, a bit each (8 instructions), then sums the set ones: a
// wavefront runs the terms about as often as its longest lane has partners.
// `near` (LDS, a column per thread): the words of bits with the LDS index of
// each word's first candidate; when they are full the partners so far are
// summed.
// Bound by FP64 issue and its latency at 3 wavefronts per SIMD (58-65% issue).
// Chimera SRK at N = 262,144: pass 1 371 -> 142 us, pass 2 499 -> 163 us; at N =
// 1000 (SE, 16 lanes per particle) 45.6 -> 12.6 us.  Also tried: candidates
// interleaved over the lanes (186 and 220 us: three address instructions per
// candidate), one partner a turn (145 and 177 us), the next turn's partners read
// ahead (151 and 174 us: more registers), 4 wavefronts per SIMD forced (spills,
// 146 and 182 us), 4 lanes at least (136 and 179 us).
constexpr int kNearWords = 8;
struct NearWords {
  uint32_t bits[kNearWords][kPairBlock];
  uint16_t first[kNearWords][kPairBlock];
};

// The run [a, b) of lane g among `len` candidates.
__device__ __forceinline__ void lane_run(int len, int g, int lg, int &a, int &b) {
  const int per = (len + (1 << lg) - 1) >> lg;
  a = min(g * per, len);
  b = min(a + per, len);
}

template <class Acc>
__device__ __forceinline__ int visit_lds64(Acc &acc, const Src64 &src, const SegShared &sh, int ncol, int qi, int ei,
                                           int g, bool wraps, NearWords *near, const KParams &P) {
  const int lg = __builtin_ctz((unsigned)P.lanes);
  int cand = 0;
#pragma unroll
  for (int r = 0; r < 3; ++r) cand += sh.off[r * ncol + qi + 2] - sh.off[r * ncol + qi - 1];
  const auto row_run = [&](int r, int &m0, int &hi) {
    const int lo = sh.off[r * ncol + qi - 1];
    int a, b;
    lane_run(sh.off[r * ncol + qi + 2] - lo, g, lg, a, b);
    m0 = lo + a;
    hi = lo + b;
  };
  if constexpr (HasNear<Acc>::value) {
    const int me = threadIdx.x;
    CohQueue64 cq;
    int r = 0, m0, hi;
    row_run(0, m0, hi);
    bool more = true;  // candidates left (of any lane)
    while (more) {
      int words = 0;
      while (words < kNearWords) {
        while (m0 >= hi && r < 2) {
          ++r;
          row_run(r, m0, hi);
        }
        if (m0 >= hi) break;
        const int cnt = min(32, hi - m0);
        uint32_t word = 0;
        // four at a time; those past the run (read from the LDS that follows)
        // are masked off
        for (int u = 0; u < cnt; u += 4) {
          uint32_t b = 0;
          if (wraps) {
#pragma unroll
            for (int k = 0; k < 4; ++k) b |= acc.template near<true>(src, m0 + u + k, P) ? 1u << k : 0u;
          } else {
#pragma unroll
            for (int k = 0; k < 4; ++k) b |= acc.template near<false>(src, m0 + u + k, P) ? 1u << k : 0u;
          }
          word |= b << u;
        }
        if (cnt < 32) word &= (1u << cnt) - 1u;
        if ((unsigned)(ei - m0) < 32u) word &= ~(1u << (ei - m0));  // not the particle itself
        near->bits[words][me] = word;
        near->first[words][me] = (uint16_t)m0;
        ++words;
        m0 += 32;
      }
      more = __any(m0 < hi || r < 2);
      // the set bits in turn, the wavefront's lanes in step, two partners (of one
      // word) a turn; the cohesion queue is emptied when it may overflow and after
      // the last partner
      using In = typename Acc::In;
      uint32_t m = 0;
      int w = 0, first = 0;
      bool left = true;
      while (left) {
        if (m == 0 && w < words) {  // (an empty word leaves the lane idle for a turn)
          m = near->bits[w][me];
          first = near->first[w][me];
          ++w;
        }
        if (m != 0) {
          const int c0 = first + __builtin_ctz(m);
          m &= m - 1u;
          const bool two = m != 0;
          const int c1 = two ? first + __builtin_ctz(m) : c0;
          m &= m - 1u;  // (0 stays 0)
          const In v0(src, c0), v1(src, c1);
          const bool q0 = acc.template term<true>(v0, true, P), q1 = acc.template term<true>(v1, two, P);
          if (q0) cq.push(c0);
          if (q1) cq.push(c1);
        }
        left = __any(m != 0 || w < words);
        if (!left || __any(cq.n > CohQueue64::kFull - 2)) cq.drain(acc, src, P);
      }
    }
  } else {
#pragma unroll 1
    for (int r = 0; r < 3; ++r) {
      int m0, hi;
      row_run(r, m0, hi);
#pragma unroll 2
      for (int m = m0; m < hi; ++m)
        if (m != ei) acc.pair(src, m, P);
    }
  }
  return cand - 1;
}

// The FP32 vortex pass 2: as visit_lds64, one lane to a particle.  Its term (60
// instructions, and the cohesion's) stood behind the distance test, where nearly
// every candidate of a wavefront ran it for the third of the lanes that needed it;
// the partners' terms, and their order in each sum, are visit_lds's.  Two partners'
// terms are formed together: at the sizes of one replica a SIMD holds one wavefront,
// and the chain of operations bounds it.  N = 1000: 48 -> 33
// us, N = 50,000: 51 -> 39, N = 400,000: 118 -> 109.  In cells of fewer than
// kNearPerCell = 42 particles: in fuller ones a wavefront's lanes lie in one cell and
// read the same candidates at once, which visit_lds does from one LDS address.  An SRK
// step on 50 x 50 cells with visit_lds and so: 81 and 69 us at 10 per cell, 154 and 149
// at 30, 189 and 192 at 40, 295 and 409 at 60, 1245 and 1393 at 130; on 10 x 10 cells
// 159 and 149 at 37, 179 and 179 at 45, 211 and 217 at 55.
template <class Acc>
__device__ __forceinline__ void visit_near32(Acc &acc, const Src32 &src, const SegShared &sh, int ncol, int qi, int ei,
                                             NearWords *near, const KParams &P) {
  const int me = threadIdx.x;
  const float lim = fmaxf(P.rho2f_hi, P.xr2f_hi);  // beyond it no decision finds a partner
  const float ol = acc.co.col(-1), oc = acc.co.col(0), orr = acc.co.col(1);
  struct Row {  // a stencil row's columns and offset, for the candidates from `first` on
    int b1, b2;
    float oy;
  };
  const auto row = [&](int r) {
    return Row{sh.off[r * ncol + qi], sh.off[r * ncol + qi + 1], (float)(r - 1) * P.hyf - acc.yl};
  };
  const auto row_of = [&](int m) { return row((m >= sh.off[ncol]) + (m >= sh.off[2 * ncol])); };
  const auto ox = [&](const Row &w, int m) { return m < w.b1 ? ol : (m >= w.b2 ? orr : oc); };
  CohQueue64 cq;
  int r = 0, m0 = sh.off[qi - 1], hi = sh.off[qi + 2];
  Row at = row(0);
  bool more = true;
  while (more) {
    int words = 0;
    while (words < kNearWords) {
      while (m0 >= hi && r < 2) {
        ++r;
        m0 = sh.off[r * ncol + qi - 1];
        hi = sh.off[r * ncol + qi + 2];
        at = row(r);
      }
      if (m0 >= hi) break;
      const int cnt = min(32, hi - m0);
      uint32_t word = 0;
      for (int u = 0; u < cnt; u += 4) {  // those past the run are masked off
        uint32_t b = 0;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const float2 v = *(const float2 *)(src.f4 + m0 + u + k);
          const float dx = v.x + ox(at, m0 + u + k), dy = v.y + at.oy;
          b |= __builtin_fmaf(dx, dx, dy * dy) <= lim ? 1u << k : 0u;
        }
        word |= b << u;
      }
      if (cnt < 32) word &= (1u << cnt) - 1u;
      if ((unsigned)(ei - m0) < 32u) word &= ~(1u << (ei - m0));  // not the particle itself
      near->bits[words][me] = word;
      near->first[words][me] = (uint16_t)m0;
      ++words;
      m0 += 32;
    }
    more = __any(m0 < hi || r < 2);
    uint32_t m = 0;
    int w = 0, first = 0;
    Row in = at;
    bool left = true;
    while (left) {
      if (m == 0 && w < words) {
        m = near->bits[w][me];
        first = near->first[w][me];
        in = row_of(first);
        ++w;
      }
      if (m != 0) {
        const int c0 = first + __builtin_ctz(m);
        m &= m - 1u;
        const bool two = m != 0;
        const int c1 = two ? first + __builtin_ctz(m) : c0;
        m &= m - 1u;  // (0 stays 0)
        const float4 v0 = src.f4[c0], v1 = src.f4[c1];
        const float a0 = src.aj[c0], a1 = src.aj[c1];
        const float dx0 = v0.x + ox(in, c0), dy0 = v0.y + in.oy, dx1 = v1.x + ox(in, c1), dy1 = v1.y + in.oy;
        const float s0 = __builtin_fmaf(dx0, dx0, dy0 * dy0), s1 = __builtin_fmaf(dx1, dx1, dy1 * dy1);
        bool inr0, inc0, inn0, inr1, inc1, inn1;
        acc.decide(src, c0, s0, inr0, inc0, inn0, P);
        acc.decide(src, c1, s1, inr1, inc1, inn1, P);
        const auto t0 = acc.align(v0, dx0, dy0, s0, inn0, a0, P), t1 = acc.align(v1, dx1, dy1, s1, inn1, a1, P);
        if (inr0) {
          acc.A0.add_prod(t0.w, t0.cph);
          acc.A1.add(t0.t);
        }
        if (inr1 & two) {
          acc.A0.add_prod(t1.w, t1.cph);
          acc.A1.add(t1.t);
        }
        if (inc0) cq.push(c0);
        if (inc1 & two) cq.push(c1);
      }
      left = __any(m != 0 || w < words);
      if (!left || __any(cq.n > CohQueue64::kFull - 2)) {
        while (cq.n > 0) {
          --cq.n;
          const int c = (int)((cq.q >> (16 * cq.n)) & 0xffffu);
          const Row z = row_of(c);
          const float4 v = src.f4[c];
          const float dx = v.x + ox(z, c), dy = v.y + z.oy;
          acc.cohesion(src, c, v, dx, dy, __builtin_fmaf(dx, dx, dy * dy), P);
        }
      }
    }
  }
}

// A candidate's values in registers, read by an accumulator as element 0.  The global
// FP64 walk requests them a candidate ahead: with several lanes to a particle its
// loads touch as many cache lines at once, and of two latencies per candidate (the
// position, then a partner's phase) none but the first is left in the open.  An SRK
// step with half of 20,000 chimera particles in one cell 457 -> 291 ms (one lane to a
// particle, nothing ahead: 304), vortex arrays 1330 -> 1223 (1091); with half of
// 200,000 in 100 spots 32 -> 23 (30) and 42 -> 40 (48).  Two ahead: the same.
struct Values {
  double x, y, p, c, s, aj;
  template <class Acc>
  __device__ __forceinline__ void load(const Src64 &g, int m) {
    x = g.x[m];
    y = g.y[m];
    if constexpr (HasNear<Acc>::value) {
      p = g.p[m];
    } else {
      c = g.c[m];
      s = g.s[m];
    }
    if (g.aj) aj = g.aj[m];
  }
  __device__ __forceinline__ Src64 src() const { return Src64{&x, &y, &p, &c, &s, &aj}; }
};
// Same visit over the global tiles, cell by cell (slot k in cell c); the FP64
// forms' lane g takes the run of each stencil row that visit_lds64 gives it.
template <class Acc, class S>
__device__ __forceinline__ int visit_global(Acc &acc, const S &src, const int *start, int c, int k, int g,
                                            const KParams &P) {
  const int cx = c % P.nx, cy = c / P.nx;
  int cand = 0;
  for (int dyo = -1; dyo <= 1; ++dyo) {
    const int row = adjust_cell(cy + dyo, P.ny) * P.nx;
    int pos = 0, ra = 0, rb = 0;  // the row's candidates before this cell; the lane's run of the row
    if constexpr (!std::is_same<S, Src32>::value) {
      int len = 0;
      for (int dxo = -1; dxo <= 1; ++dxo) {
        const int jc = row + adjust_cell(cx + dxo, P.nx);
        len += start[jc + 1] - start[jc];
      }
      lane_run(len, g, __builtin_ctz((unsigned)P.lanes), ra, rb);
    }
    for (int dxo = -1; dxo <= 1; ++dxo) {
      const int jc = row + adjust_cell(cx + dxo, P.nx);
      const int m0 = start[jc], m1 = start[jc + 1];
      // column offsets from the boundary trick: all of [m0, m1) is one column
      if (dxo < 0) acc.row(dyo, m1, m1, P);
      else if (dxo == 0) acc.row(dyo, m0, m1, P);
      else acc.row(dyo, m0, m0, P);
      cand += m1 - m0;
      if constexpr (std::is_same<S, Src32>::value) {
        // per cell FP32 partials, as visit_lds sums them
        acc.cell_begin();
        for (int m = m0; m < m1; ++m)
          if (m != k) acc.template pair<SUM_GROUP>(src, m, P);
        acc.flush();
      } else {
        const int b = m0 + max(0, ra - pos), e = m0 + min(m1 - m0, rb - pos);
        if (b < e) {
          Values v, next;
          next.load<Acc>(src, b);
#pragma unroll 1
          for (int m = b; m < e; ++m) {
            v = next;
            next.load<Acc>(src, min(m + 1, e - 1));
            if (m != k) acc.pair(v.src(), 0, P);
          }
        }
        pos += m1 - m0;
      }
    }
  }
  return cand - 1;
}

// A halo column or row of the workgroup wraps: without one the candidates'
// separations need no min-image.  A candidate is less than two cells away along an
// axis, so that with four cells or more the plain difference is the nearer image;
// with three it may lie beyond half the box, and a cutoff wider than a cell (xi_r)
// then finds its nearer image.
__device__ __forceinline__ bool wraps(const KParams &P, const Seg &g) {
  return g.cx0 < 1 || g.cx0 + g.W >= P.nx || g.cy < 1 || g.cy + 1 >= P.ny || P.nx < 4 || P.ny < 4;
}

// The words of the walks that find the near partners first, after the staged tiles.
template <int PREC, int PASS>
__device__ __forceinline__ NearWords *near_words(void *dyn_lds, const KParams &P) {
  return (NearWords *)((char *)dyn_lds + (size_t)P.lds_cap * LdsTile<PREC, PASS>::bytes);
}

// =============================================================================
// Pass-1 and pass-2 kernels over linked cells
// =============================================================================

template <class Acc, int PREC, int EPI>
__device__ __forceinline__ void pass1_segment(const KParams &P, const int *__restrict__ start, const Tiles &t,
                                              const int *__restrict__ slot_h, const int *__restrict__ slot_id,
                                              const double *gp, const EpiCtx &e, unsigned long long *counts, int seg,
                                              SegShared &sh, void *dyn_lds) {
  Block b;
  if (!block_range(P, start, t, seg, b)) return;  // the whole workgroup
  const bool fits = b.W <= kMaxSegW;
  Seg g{};
  if (fits) g = halo_setup(P, start, b.cy, b.cx0, b.W, sh);
  bool staged = fits && g.total <= P.lds_cap;
  LdsTile<PREC, 1> lt(dyn_lds, P.lds_cap);
  bool fit = true;  // phases (and alpha) the staged walk's sine takes
  if (staged) {
    for (int el = threadIdx.x; el < g.total; el += kPairBlock) {
      int s = find_slot(sh, g.ns, el);
      lt.load(el, sh.gst[s] + (el - sh.off[s]), t, e);
      if constexpr (PREC == P64) fit &= phase_fits(lt.a[el]);
    }
  }
  if constexpr (PREC == P64)
    staged = __syncthreads_and(staged && fit && phase_fits(P.alpha));
  else
    __syncthreads();
  // the centre slots are contiguous from the first centre cell's, k0 its slot
  // (k0 - gst) of the cell
  const int e0 = staged ? sh.off[g.ncol + 1] + (b.k0 - sh.gst[g.ncol + 1]) : 0;
  const int ncen = b.k1 - b.k0;
  const int k0 = b.k0;
  // FP64 forms: P.lanes lanes per particle, lane 0 of them writes it
  const int lg = PREC == P32K ? 0 : __builtin_ctz((unsigned)P.lanes), gl = threadIdx.x & ((1 << lg) - 1);
  long long cand_sum = 0, n_sum = 0, n2_sum = 0;
  for (int p = threadIdx.x >> lg; p < ncen; p += kPairBlock >> lg) {
    const int k = k0 + p, ei = e0 + p;
    Acc acc;
    int cand;
    if (staged) {
      int lo = 1, hi = g.W;  // centre column of ei
      while (lo < hi) {
        int mid = (lo + hi + 1) >> 1;
        if (sh.off[g.ncol + mid] <= ei) lo = mid;
        else hi = mid - 1;
      }
      acc.init(lt.src(), ei, k, t, P);
      if constexpr (PREC == P32K)
        cand = visit_lds(acc, lt.src(), sh, g.ncol, lo, ei, P);
      else
        cand = visit_lds64(acc, lt.src(), sh, g.ncol, lo, ei, gl, wraps(P, g), near_words<PREC, 1>(dyn_lds, P), P);
    } else {
      auto gs = global_src<PREC>(t, e, 1);
      acc.init(gs, k, k, t, P);
      cand = visit_global(acc, gs, start, t.cell[k], k, gl, P);
    }
    if constexpr (PREC != P32K) {
      acc.reduce(P.lanes);
      if (gl) continue;  // lane 0 of the particle's lanes writes it
    }
    const int h = slot_h[k], id = slot_id[k];
    Pass1Out o{};
    acc.finish(P, PREC == P32K ? gp[h] : 0.0, o);
    bin_stage<EPI>(P, e, h, id, epilogue1<EPI>(P, e, h, id, k, o));
    cand_sum += cand;
    n_sum += o.n;
    n2_sum += o.n2;
  }
  if (counts) count_add(counts, cand_sum, n_sum, n2_sum);
}

template <class Acc, int PREC, int EPI>
__device__ __forceinline__ void pass2_segment(const KParams &P, const int *__restrict__ start, const Tiles &t,
                                              const int *__restrict__ slot_h, const int *__restrict__ slot_id,
                                              const double *gp, const EpiCtx &e, int seg, SegShared &sh, void *dyn_lds) {
  Block b;
  if (!block_range(P, start, t, seg, b)) return;
  const bool fits = b.W <= kMaxSegW;
  Seg g{};
  if (fits) g = halo_setup(P, start, b.cy, b.cx0, b.W, sh);
  bool staged = fits && g.total <= P.lds_cap;
  LdsTile<PREC, 2> lt(dyn_lds, P.lds_cap);
  bool fit = true;  // phases (and alpha) the staged walk's sine takes
  if (staged) {
    for (int el = threadIdx.x; el < g.total; el += kPairBlock) {
      int s = find_slot(sh, g.ns, el);
      lt.load(el, sh.gst[s] + (el - sh.off[s]), t, e);
      if constexpr (PREC == P64) fit &= phase_fits(lt.a[el]);
    }
  }
  if constexpr (PREC == P64)
    staged = __syncthreads_and(staged && fit && phase_fits(P.alpha));
  else
    __syncthreads();
  const int e0 = staged ? sh.off[g.ncol + 1] + (b.k0 - sh.gst[g.ncol + 1]) : 0;
  const int ncen = b.k1 - b.k0;
  const int k0 = b.k0;
  const int lg = PREC == P32K ? 0 : __builtin_ctz((unsigned)P.lanes), gl = threadIdx.x & ((1 << lg) - 1);
  for (int p = threadIdx.x >> lg; p < ncen; p += kPairBlock >> lg) {
    const int k = k0 + p, ei = e0 + p;
    const int h = slot_h[k], id = slot_id[k];
    Pass2In in{e.aphi_slot[k], e.n_slot[k], e.n2_slot[k], 0.0, 0.0};
    if (EPI == EPI_ITO2) {
      in.in0 = e.a0[h];
      in.in1 = e.a1[h];
    }
    Acc acc;
    if (staged) {
      int lo = 1, hi = g.W;
      while (lo < hi) {
        int mid = (lo + hi + 1) >> 1;
        if (sh.off[g.ncol + mid] <= ei) lo = mid;
        else hi = mid - 1;
      }
      acc.init(lt.src(), ei, k, t, P, in);
      bool near = false;
      if constexpr (HasNear32<Acc>::value) {
        near = P.near[1] != 0;
        if (near) visit_near32(acc, lt.src(), sh, g.ncol, lo, ei, near_words<PREC, 2>(dyn_lds, P), P);
      }
      if constexpr (PREC == P32K) {
        if (!near) visit_lds(acc, lt.src(), sh, g.ncol, lo, ei, P);
      } else {
        visit_lds64(acc, lt.src(), sh, g.ncol, lo, ei, gl, wraps(P, g), near_words<PREC, 2>(dyn_lds, P), P);
      }
    } else {
      auto gs = global_src<PREC>(t, e, 2);
      acc.init(gs, k, k, t, P, in);
      visit_global(acc, gs, start, t.cell[k], k, gl, P);
    }
    if constexpr (PREC != P32K) {
      acc.reduce(P.lanes);
      if (gl) continue;
    }
    Pass2Out o;
    acc.finish(P, PREC == P32K ? gp[h] : 0.0, o);
    epilogue2<EPI>(P, e, h, id, o);
  }
}

}  // namespace
}  // namespace spc2
