// Single-system pair kernels on gfx950 (chimera and vortex arrays): the
// linked-cell kernels over the row-segment LDS staging of spc2_lds_stencil.h,
// the all-pairs path, and their dispatch.  Compiled with -ffp-contract=off.
#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdlib>

#include "spc2_device.h"
#include "spc2_internal.h"
#include "spc2_chimera_mfma.h"
#include "spc2_lds_stencil.h"

namespace spc2 {

namespace {

constexpr int kBlock = 256;

inline int blocks_for(long long n, int b = kBlock) { return (int)((n + b - 1) / b); }

// =============================================================================
// Pass-1 and pass-2 kernels over linked cells
// =============================================================================

// (FP64: three wavefronts per SIMD at the least, for which the vortex passes keep 4 to
// 33 registers in scratch.  With two, N = 160,000: 86 us for 76 of RK4's pass; N =
// 100,000, SRK: 50 for 52 and 91 for 89.  FP32 pass 1: four, which the vortex passes
// that bin their next stage miss by 3 to 5 registers: 153 for 130 us at N = 1M, where
// the bin kernel of its own takes 17 and the pass without it 117.)
template <class Acc, int PREC, int EPI>
__global__ __launch_bounds__(kBlock)
__attribute__((amdgpu_waves_per_eu(PREC == P64 ? 3 : (PREC == P32K ? 4 : 1)))) void k_pass1_lds(KParams P, const int *__restrict__ start, Tiles t,
                                                      const int *__restrict__ slot_h, const int *__restrict__ slot_id,
                                                      const double *gp, EpiCtx e, unsigned long long *counts) {
  extern __shared__ float4 dyn_lds[];
  __shared__ SegShared sh;
  pass1_segment<Acc, PREC, EPI>(P, start, t, slot_h, slot_id, gp, e, counts, xcd_segment(blockIdx.x, gridDim.x),
                                sh, dyn_lds);
}

template <class Acc, int PREC, int EPI>
__global__ __launch_bounds__(kBlock)
__attribute__((amdgpu_waves_per_eu(PREC == P64 ? 3 : 1))) void k_pass2_lds(KParams P, const int *__restrict__ start, Tiles t,
                                                      const int *__restrict__ slot_h, const int *__restrict__ slot_id,
                                                      const double *gp, EpiCtx e) {
  extern __shared__ float4 dyn_lds[];
  __shared__ SegShared sh;
  pass2_segment<Acc, PREC, EPI>(P, start, t, slot_h, slot_id, gp, e, xcd_segment(blockIdx.x, gridDim.x), sh, dyn_lds);
}

// The matrix-core passes of dense FP32 chimera cells.
template <int EPI, bool SHORT>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(3))) void k_pass1_mfma(KParams P, const int *__restrict__ start, Tiles t,
                                                       const int *__restrict__ slot_h, const int *__restrict__ slot_id,
                                                       const double *gp, EpiCtx e, unsigned long long *counts) {
  extern __shared__ float4 dyn_lds[];
  __shared__ SegShared sh;
  mfma_segment<1, EPI, SHORT>(P, start, t, slot_h, slot_id, gp, e, counts, xcd_segment(blockIdx.x, gridDim.x), sh, dyn_lds);
}

template <int EPI, bool SHORT>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(3))) void k_pass2_mfma(KParams P, const int *__restrict__ start, Tiles t,
                                                       const int *__restrict__ slot_h, const int *__restrict__ slot_id,
                                                       const double *gp, EpiCtx e) {
  extern __shared__ float4 dyn_lds[];
  __shared__ SegShared sh;
  mfma_segment<2, EPI, SHORT>(P, start, t, slot_h, slot_id, gp, e, nullptr, xcd_segment(blockIdx.x, gridDim.x), sh, dyn_lds);
}

// =============================================================================
// All pairs (rho > L/4): a wavefront per particle (allpairs_pass1), four to a
// workgroup.
// =============================================================================

template <int PREC, int SYS, int EPI>
__global__ __launch_bounds__(kBlock) void k_pass1_allpairs(KParams P, const double *gx, const double *gy,
                                                           const double *gp, const float4 *tiles, EpiCtx e,
                                                           unsigned long long *counts) {
  const int i = blockIdx.x * (kBlock / kApLanes) + threadIdx.x / kApLanes, g = threadIdx.x % kApLanes;
  const bool active = i < P.n, lead = active && g == 0;  // whole wavefronts
  Pass1Out o{};
  if (active) {
    allpairs_pass1<PREC, SYS>(P, i, g, gx, gy, gp, tiles, o);
    if (lead) stage_next<EPI>(e, i, epilogue1<EPI>(P, e, i, i, i, o));  // all pairs: home order is the id order
  }
  if (counts) count_add(counts, lead ? P.n - 1 : 0, lead ? o.n : 0, lead ? o.n2 : 0);
}

template <int SYS, int EPI>
__global__ __launch_bounds__(kBlock) void k_pass2_allpairs(KParams P, const double *gx, const double *gy,
                                                           const double *gp, EpiCtx e) {
  const int i = blockIdx.x * (kBlock / kApLanes) + threadIdx.x / kApLanes, g = threadIdx.x % kApLanes;
  if (i >= P.n) return;  // whole wavefronts
  Pass2Out o;
  const double in0 = EPI == EPI_ITO2 ? e.a0[i] : 0.0, in1 = EPI == EPI_ITO2 ? e.a1[i] : 0.0;
  allpairs_pass2<SYS>(P, i, g, gx, gy, gp, e.aphi_slot, e.n_slot, e.n2_slot, in0, in1, o);
  if (g == 0) stage_next<EPI>(e, i, epilogue2<EPI>(P, e, i, i, o));
}

// =============================================================================
// dispatch
// =============================================================================

// Has the launch write the next stage (s.vnext, consumed here): the bins of linked
// cells, or the all-pairs path's second stage arrays.
bool take_next(Sim &s, EpiCtx &e) {
  if (!s.vnext) return false;
  e.next = s.vnext;
  e.kcdt_n = s.vnext_kcdt;
  s.vnext = 0;
  if (s.linked) {
    e.bgx = s.gx;
    e.bgy = s.gy;
    e.bgp = s.gp;
    e.bins = s.bins();
  } else {
    e.bgx = s.gx2;
    e.bgy = s.gy2;
    e.bgp = s.gp2;
    e.tn.f4 = s.t2.f4;
  }
  return true;
}

void next_taken(Sim &s) {
  if (!s.linked) {
    std::swap(s.gx, s.gx2);
    std::swap(s.gy, s.gy2);
    std::swap(s.gp, s.gp2);
    std::swap(s.t.f4, s.t2.f4);
  }
  s.staged = true;
}

template <int PREC, int SYS, int EPI>
void pass1_typed(Sim &s, const EpiCtx &e) {
  unsigned long long *cnt = s.counting ? s.counts : nullptr;
  if (s.linked) {
    const dim3 grid(s.ny * s.kp.segs), blk(kBlock);
    const size_t sh = pair_lds_bytes(s.kp, PREC, 1);
    if constexpr (PREC == P32K && SYS == SPC2_CHIMERA) {
      if (s.kp.mfma) {
        launch_pair(s, s.kp.chunk <= kMfmaShort ? k_pass1_mfma<EPI, true> : k_pass1_mfma<EPI, false>, grid, blk, sh, s.kp, (const int *)s.start, s.t, (const int *)s.slot_h,
                    (const int *)s.slot_id, (const double *)s.gp, e, cnt);
        return;
      }
    }
    if (SYS == SPC2_CHIMERA)
      launch_pair(s, k_pass1_lds<ChimAcc<PREC>, PREC, EPI>, grid, blk, sh, s.kp, (const int *)s.start, s.t,
                  (const int *)s.slot_h, (const int *)s.slot_id, (const double *)s.gp, e, cnt);
    else
      launch_pair(s, k_pass1_lds<VortAcc<PREC>, PREC, EPI>, grid, blk, sh, s.kp, (const int *)s.start, s.t,
                  (const int *)s.slot_h, (const int *)s.slot_id, (const double *)s.gp, e, cnt);
  } else {
    // the FP32 form reads cos and sin of phi_j from the stage's tiles
    launch_pair(s, k_pass1_allpairs<PREC, SYS, EPI>, dim3(blocks_for((long long)s.n * kApLanes)),
                dim3(kBlock), 0, s.kp,
                (const double *)s.gx, (const double *)s.gy, (const double *)s.gp,
                PREC == P32K ? (const float4 *)s.t.f4 : nullptr, e, cnt);
  }
}

template <int PREC, int SYS>
void pass1_epi(Sim &s, int epi, const EpiCtx &e) {
  switch (epi) {
    case EPI_K: pass1_typed<PREC, SYS, EPI_K>(s, e); break;
    case EPI_ITO1: pass1_typed<PREC, SYS, EPI_ITO1>(s, e); break;
    case EPI_SE: pass1_typed<PREC, SYS, EPI_SE>(s, e); break;
    case EPI_RK4_FINAL: pass1_typed<PREC, SYS, EPI_RK4_FINAL>(s, e); break;
  }
}

template <int PREC>
void pass1_sys(Sim &s, int epi, const EpiCtx &e) {
  if (s.P.system == SPC2_CHIMERA)
    pass1_epi<PREC, SPC2_CHIMERA>(s, epi, e);
  else
    pass1_epi<PREC, SPC2_VORTEX>(s, epi, e);
}

template <int PREC, int SYS, int EPI>
void pass2_typed(Sim &s, const EpiCtx &e) {
  if (s.linked) {
    const size_t sh = pair_lds_bytes(s.kp, PREC, 2);
    const dim3 grid(s.ny * s.kp.segs), blk(kBlock);
    if constexpr (PREC == P32K && SYS == SPC2_CHIMERA) {
      if (s.kp.mfma) {
        launch_pair(s, s.kp.chunk <= kMfmaShort ? k_pass2_mfma<EPI, true> : k_pass2_mfma<EPI, false>, grid, blk, sh, s.kp, (const int *)s.start, s.t, (const int *)s.slot_h,
                    (const int *)s.slot_id, (const double *)s.gp, e);
        return;
      }
    }
    if (SYS == SPC2_CHIMERA)
      launch_pair(s, k_pass2_lds<Chim2Acc<PREC>, PREC, EPI>, grid, blk, sh, s.kp, (const int *)s.start, s.t,
                  (const int *)s.slot_h, (const int *)s.slot_id, (const double *)s.gp, e);
    else
      launch_pair(s, k_pass2_lds<Vort2Acc<PREC>, PREC, EPI>, grid, blk, sh, s.kp, (const int *)s.start, s.t,
                  (const int *)s.slot_h, (const int *)s.slot_id, (const double *)s.gp, e);
  } else {
    launch_pair(s, k_pass2_allpairs<SYS, EPI>, dim3(blocks_for((long long)s.n * kApLanes)), dim3(kBlock), 0, s.kp, (const double *)s.gx,
                (const double *)s.gy, (const double *)s.gp, e);
  }
}

template <int PREC, int SYS>
void pass2_epi(Sim &s, int epi, const EpiCtx &e) {
  if (epi == EPI_ITO2)
    pass2_typed<PREC, SYS, EPI_ITO2>(s, e);
  else
    pass2_typed<PREC, SYS, EPI_SRK>(s, e);
}

template <int PREC>
void pass2_sys(Sim &s, int epi, const EpiCtx &e) {
  if (s.P.system == SPC2_CHIMERA)
    pass2_epi<PREC, SPC2_CHIMERA>(s, epi, e);
  else
    pass2_epi<PREC, SPC2_VORTEX>(s, epi, e);
}

constexpr int kLanes64 = 2;
constexpr long long kLanesFill = 131072;
constexpr double kLanesPerCell[2] = {0.85, 1.5};  // chimera, vortex arrays
constexpr double kDensePerCell = 170.0;
constexpr int kDenseN = 16384;
constexpr double kMfmaPerCell = 20.0;
constexpr double kNearPerCell = 42.0;

// bytes per staged candidate of the larger pass
int lds_elem_bytes(int prec) {
  switch (prec) {
    case P32K: return LdsTile<P32K, 2>::bytes;
    case P64: return LdsTile<P64, 2>::bytes;
    default: return LdsTile<P64F, 2>::bytes;
  }
}

}  // namespace

// Candidates of a matrix-core workgroup at the most, and what the rows' padding and
// the far tile take of them: 76 KB of LDS, two workgroups of pass 2 per CU as with 60.
// Chunks are kept to kMfmaHalo candidates where they can be, three workgroups of pass
// 1 per CU (past it, SRK steps at 150 to 160 particles per cell take 10 to 19% longer).
constexpr int kMfmaLdsBytes = 76 * 1024;
constexpr int kMfmaCap = (kMfmaLdsBytes - MfmaLds<2>::tail_bytes) / MfmaLds<2>::tile_bytes * kMfmaTile;
constexpr int kMfmaHalo = 2752;
constexpr double kMfmaPad = 128.0;

// its mean halo with a margin, for a chunk of row slots: the chunk's cells, a partial
// cell at each end and the sides, padded
static double mfma_halo(int chunk, double per_cell) {
  return 1.25 * 3.0 * (chunk + 3.0 * per_cell) + kMfmaPad;
}

// a row's mean count and four standard deviations, in chunks
static int chunks_per_row(const KParams &k) {
  const double row = (double)k.n / (double)k.ny;
  return std::max(1, (int)std::ceil((row + 4.0 * std::sqrt(row) + 8.0) / k.chunk));
}

// The pair workgroups of a linked system: about `target` lanes each and an LDS
// capacity for their halo.
// * The FP64 forms split each particle's candidates over `lanes` lanes: enough
//   for kLanesFill lanes in all (two wavefronts on each of the 1024 SIMDs), at
//   most 16, so that small systems fill the device; the plain form at least
//   kLanes64, whose halved workgroups leave room for its words of bits.  The
//   count depends on the system alone, so that a batch's replica sums as a single
//   handle does.  In sparse cells no more lanes than kLanesPerCell times the mean
//   filling: a stencil row of three cells has little for more, and a batch, which
//   fills the device by itself, pays for their workgroups (64 chimera replicas of N
//   = 2000, SRK step, 16 lanes and so: plain 348 and 123 us at 1 per cell, 367 and
//   103 at 2, 382 and 152 at 4, 335 and 198 at 7; alone 39 and 29, 38 and 30, 37 and
//   38, 38 and 40; one lane of the library's sines: 148 to 219).  Nor in cells from
//   kDensePerCell particles on, of systems of at least kDenseN, where no halo is
//   staged whatever the lanes and their loads of different candidates at once cost
//   more than they gain (chimera SRK step in 10 x 10 and 14 x 14 cells of 200, with 8
//   and 4 lanes: plain 612 and 1044 us, so 650 and 820; factored 686 and 1135, so 586
//   and 599).
// * Rows of at least kChunkPerCell particles per cell are cut into chunks of
//   `target` slots rounded to whole wavefronts, so that every wavefront but a
//   row's last is full.  A row gets workgroups for its mean count plus four
//   standard deviations; its last workgroup takes whatever remains.
// * Sparser rows are cut into segments of seg_w cells (at most kMaxSegW), whose
//   particle counts follow the cells.
// The LDS capacity is the mean halo with a margin, within 60 KB; a workgroup
// whose halo exceeds it reads the same tiles from global memory.
// * The FP32 chimera form of rows with at least kMfmaPerCell particles per cell
//   takes the matrix-core passes, whose LDS holds whole tiles, within 76 KB.  Where
//   the halo of a chunk does not fit, the chunk is halved, to 32 slots at the least;
//   where the two or so cells that such a chunk touches have too many neighbours for
//   it (from 214 particles per cell on), the scalar walk of the FP32 form is the
//   faster one.  An SRK step, before (chunks of 256 within 60 KB, every filling) and
//   so, with the scalar walk's time: in 16 x 16 cells 94 and 94 us (235) at 160 per
//   cell, 950 and 104 (683) at 180, 1091 and 123 (735) at 200; in 50 x 50 cells 885
//   and 340 (486) at 130, 3933 and 759 (1877) at 200; past the line, on the matrix
//   cores all the same, 6360 (4979) at 280.
void configure_segments_kp(KParams &k, int prec, int system, double target) {
  k.chunk = 0;
  k.lanes = 1;
  k.mfma = 0;
  k.aj = k.raj = 1.0;
  k.bin_cap = 0;
  k.near[0] = prec == P64 ? (int)sizeof(NearWords) : 0;
  k.near[1] = prec == P64 ? (int)sizeof(NearWords) : 0;
  if (!k.linked) {
    k.seg_w = k.segs = 1;
    k.lds_cap = 0;
    return;
  }
  const double per_cell = (double)k.n / ((double)k.nx * (double)k.ny);
  if (prec != P32K) {
    const int least = prec == P64 ? kLanes64 : 1;
    const int most = per_cell >= kDensePerCell && k.n >= kDenseN ? least : 16;
    while (k.lanes < least ||
           (k.lanes < most && k.lanes < kLanesPerCell[system] * per_cell && (long long)k.n * k.lanes < kLanesFill))
      k.lanes *= 2;
  }
  target /= k.lanes;  // particles per workgroup
  if (prec == P32K && system == SPC2_VORTEX && per_cell < kNearPerCell) k.near[1] = (int)sizeof(NearWords);
  double halo;
  if (per_cell >= kChunkPerCell) {
    const int unit = 64 / k.lanes;  // a wavefront's particles
    int chunk = unit * std::max(1, (int)std::lround(target / unit));
    // at most kMaxSegW - 3 cells' worth, so a chunk's columns fit the halo tables
    chunk = std::min(chunk, unit * std::max(1, (int)std::floor((kMaxSegW - 3) * per_cell / unit)));
    k.chunk = chunk;
    k.segs = chunks_per_row(k);
    k.seg_w = std::min(k.nx, (int)std::ceil(chunk / per_cell) + 1);
    halo = 1.25 * 3.0 * (chunk + 3.0 * per_cell);  // chunk's cells, a partial cell at each end, and the sides
    // the halo of the shortest chunks: of two cells, with four standard deviations
    const double two = 12.0 * per_cell + 4.0 * std::sqrt(12.0 * per_cell) + kMfmaPad;
    if (prec == P32K && system == SPC2_CHIMERA && per_cell >= kMfmaPerCell && two <= kMfmaCap) {
      k.mfma = 1;
      k.chunk = std::min(chunk, kMfmaWindow);
      while (k.chunk > 2 * kMfmaTile && mfma_halo(k.chunk, per_cell) > kMfmaHalo) k.chunk /= 2;
      halo = std::max(mfma_halo(k.chunk, per_cell), two);
      k.segs = chunks_per_row(k);
      // |a_j| <= |sigma|: sigma times a mean of sines
      k.aj = std::exp2(std::ceil(std::log2(std::max(std::fabs(k.sigma) * 1.0001, 1e-200))));
      k.raj = 1.0 / k.aj;
    }
  } else {
    int w = (int)std::floor(target / std::max(per_cell, 1e-9));
    w = std::max(1, std::min({w, kMaxSegW, k.nx}));
    k.seg_w = w;
    k.segs = (k.nx + w - 1) / w;
    halo = 1.6 * 3.0 * (w + 2) * per_cell;
  }
  int cap;
  if (k.mfma) {
    cap = std::min(kMfmaCap, (int)std::ceil(halo / kMfmaTile) * kMfmaTile);
  } else {
    cap = (int)std::ceil((halo + 160.0) / 64.0) * 64;
    cap = std::min(cap, (kLdsBytes - k.near[1]) / lds_elem_bytes(prec));
  }
  if (const char *env = std::getenv("SPC2_LDS_CAP")) cap = std::max(0, std::min(cap, std::atoi(env)));
  k.lds_cap = k.mfma ? cap / kMfmaTile * kMfmaTile : cap;
}

size_t pair_lds_bytes(const KParams &k, int prec, int pass) {
  if (!k.linked) return 0;
  if (k.mfma) return (size_t)(pass == 1 ? MfmaLds<1>::bytes(k.lds_cap) : MfmaLds<2>::bytes(k.lds_cap));
  int elem;
  switch (prec) {
    case P32K: elem = pass == 1 ? LdsTile<P32K, 1>::bytes : LdsTile<P32K, 2>::bytes; break;
    case P64: elem = pass == 1 ? LdsTile<P64, 1>::bytes : LdsTile<P64, 2>::bytes; break;
    default: elem = pass == 1 ? LdsTile<P64F, 1>::bytes : LdsTile<P64F, 2>::bytes;
  }
  return (size_t)k.lds_cap * (size_t)elem + (size_t)k.near[pass - 1];
}

// A single handle's pair workgroups.  The matrix-core passes of a small system are
// bound by the latency of one workgroup's phases, so its chunks are halved while
// twice the workgroups still fit the device at once (four on each of 256 CUs), to 32
// slots at the least (two groups of centres).  Pass 1 of SE at N = 8191: 24.7 us with
// 256 slots, 18.7 with 128, 16.7 with 64, 14.3 with 32, 14.5 with 16; both SRK passes
// at N = 40,000: 51, 42, 39 and, past one fill, 51 with 32; at N = 120,000: 71, 67 and
// 86 with 64.  (The sums are whole numbers: no result depends on the chunk.)
void configure_segments(Sim &s) {
  KParams &k = s.kp;
  configure_segments_kp(k, s.prec, s.P.system, kSegTarget);
  if (!k.mfma) return;
  while (k.chunk > 32 && 2LL * k.n <= 1024LL * k.chunk) k.chunk /= 2;
  k.segs = chunks_per_row(k);
}

void launch_pass1(Sim &s, int epi, double *ox, double *oy, double *op, const StepArgs &sa, double *const k1[3],
                  double *const k2[3], double *const k3[3]) {
  EpiCtx e = make_ctx(s, ox, oy, op, sa, k1, k2, k3);
  const bool next = take_next(s, e);
  switch (s.prec) {
    case P64: pass1_sys<P64>(s, epi, e); break;
    case P64F: pass1_sys<P64F>(s, epi, e); break;
    default: pass1_sys<P32K>(s, epi, e);
  }
  if (next) next_taken(s);
}

void launch_pass2(Sim &s, int epi, double *a0, double *a1, const StepArgs &sa) {
  EpiCtx e = make_ctx(s, nullptr, nullptr, nullptr, sa, nullptr, nullptr, nullptr);
  e.a0 = a0;
  e.a1 = a1;
  const bool next = take_next(s, e);
  switch (s.prec) {
    case P64: pass2_sys<P64>(s, epi, e); break;
    case P64F: pass2_sys<P64F>(s, epi, e); break;
    default: pass2_sys<P32K>(s, epi, e);
  }
  if (next) next_taken(s);
}

}  // namespace spc2
