// Kernel drivers: SpMV, coloured symmetric Gauss-Seidel, fused residual +
// restriction, prolongation, the V-cycle in fp64 / fp32 / scaled fp16, and
// the vector reductions.
#include <algorithm>
#include <atomic>
#include <initializer_list>
#include <mutex>

#include "kernels.hpp"

namespace hpcgx {

static inline unsigned tiles(int64_t rows) { return (unsigned)((rows + kBlock - 1) / kBlock); }

// Steps of blocks below this many rows take one wave per workgroup on every
// level and in every precision: a block of 105105 rows is 411 workgroups of 256
// threads, so that some of the 256 CUs take two and others one, and a step lasts as
// long as the fullest.  By single waves the CUs take 6 or 7 of 1643.  SYMGS kappa
// 97x65x129 199 -> 185 us, CG on general rows 64^3 19.7 -> 18.4 ms, CG 104^3 26.5 ->
// 25.8.  Above, the split no longer shows and a workgroup's waves share the L1: up
// to 2^20 rows the fp16 V-cycle of kappa 256x192x144 (884736 rows) ran 111 -> 114 ms.
constexpr int64_t kOneWaveRows = 1 << 18;

// rz (the finest level of an fp64 stencil hierarchy only): the step also leaves the
// partials of r.x over its rows there, tiles(rows) of them.
template <class VT, class XT, class ACC, int ZK, bool FINE>
static void gs_block(Ctx *c, const Level &L, const XT *r, XT *x, int k, double *rz = nullptr) {
  const int64_t r0 = L.lay.start[k], nr = L.lay.start[k + 1] - r0;
  if (nr <= 0) return;
  const ColIdx ci = col_idx(c, L, k);
  // Coarse fp64 steps of blocks under HPCGX_ONE_WAVE_ROWS (2^20) rows launch
  // as one-wave blocks, which spreads them over more CUs: with explicit
  // columns at two waves per SIMD a 192^3 set measured 2-6 % faster, 512^3
  // about 5 %; with compact columns and no occupancy limit, 1245 against 1219
  // GFLOP/s at 192^3 (512^3 within its run-to-run spread); with paired values,
  // 94.6-95.4 ms per 192^3 set against 95.5-95.6 with the threshold at 2^16
  // (the 96^3 level's steps in 256-thread blocks) and 96.1-96.8 with none.
  // Below kOneWaveRows the fine level and the other precisions do so too; the r.z
  // form keeps 256-thread blocks.
#ifndef HPCGX_ONE_WAVE_ROWS
#define HPCGX_ONE_WAVE_ROWS (1 << 20)
#endif
  const unsigned bs = nr < kOneWaveRows || (!FINE && sizeof(VT) == 8 && nr < (int64_t)(HPCGX_ONE_WAVE_ROWS)) ? kSlice : kBlock;
  const unsigned g = (unsigned)((nr + bs - 1) / bs);
  hipStream_t st = c->stream;
  const ValSrc<VT, ACC> v = val_src<VT, ACC>(L);
  if constexpr (FINE && ZK < 0 && sizeof(VT) == 8 && sizeof(XT) == 8) {
    if (rz) {
      // 256-thread blocks: the partials are per block of 4 waves, tiles(nr) of them
      with_forms<VT, true>(L, ci, [&](auto CF, auto VF) {
        if constexpr (VF() != kValsStored) {
          if (run_rows(L, nr)) {
            k_gs_run<-1, FINE, VF(), true><<<run_tiles(nr), kBlock, 0, st>>>(ci, v, r, x, r0, nr, rz);
            return;
          }
        }
        k_gs<VT, XT, ACC, -1, FINE, CF(), VF(), false, true><<<tiles(nr), kBlock, 0, st>>>(ci, v, r, x, r0, nr, nullptr, rz);
      });
      return;
    }
  }
  if constexpr (ZK <= 0) {  // general levels: full rows, or the first block from x = 0
    if (L.dslot) {
      if (ci.cbase)
        k_gs<VT, XT, ACC, ZK, FINE, kColsSlice, kValsStored, true><<<g, bs, 0, st>>>(ci, v, r, x, r0, nr, L.dslot);
      else
        k_gs<VT, XT, ACC, ZK, FINE, kColsStored, kValsStored, true><<<g, bs, 0, st>>>(ci, v, r, x, r0, nr, L.dslot);
      return;
    }
  }
  with_forms<VT, true>(L, ci, [&](auto CF, auto VF) {
    if constexpr (VF() != kValsStored && sizeof(XT) == 8) {
      if (run_rows(L, nr)) {
        const unsigned rbs = nr < kOneWaveRows ? kSlice : kBlock;
        k_gs_run<ZK, FINE, VF()><<<run_tiles(nr, rbs), rbs, 0, st>>>(ci, v, r, x, r0, nr);
        return;
      }
    }
    k_gs<VT, XT, ACC, ZK, FINE, CF(), VF()><<<g, bs, 0, st>>>(ci, v, r, x, r0, nr, nullptr);
  });
}

// Whether steps on blocks whose classes differ in x alone share a launch
// (k_gs_lines).  They must lie at one distance per slot (has_block_offs: even extents
// in x and y, so the lines of the two blocks are alike).  Blocks of up to
// 2^18 rows: the pairs of a 104^3 and a 128^3 fine level (140608 and 262144 rows)
// gain 23 and 15 us a V-cycle, those of 192^3 (884736) lose 90.
static bool lines_pay(const Ctx *c, const Level &L) {
  return L.boffs && col_idx(c, L, 0).off && L.lay.start[1] <= (1 << 18) && L.lay.nx / 2 <= kBlock;
}

// Whether steps on blocks whose classes differ in z alone do (k_gs_columns): an even
// extent in z, so the blocks have the same planes, and at least 4 columns of
// them in a workgroup.  Blocks of up to 2^16 rows: 32768 rows gain 3 us a pair,
// 110592 lose 3 (a workgroup's columns are then a few short pieces of lines).
static bool columns_pay(const Ctx *c, const Level &L) {
  return L.boffs && col_idx(c, L, 0).off && L.lay.start[1] <= (1 << 16) && L.lay.nz % 2 == 0 &&
         L.lay.nz / 2 <= kBlock / 4;
}

// Steps of blocks a, b (STEPS 3: and a again), whose classes differ in x alone.
template <class VT, class XT, class ACC, int ZA, int ZB, int STEPS, bool FINE>
static void gs_lines(Ctx *c, const Level &L, const XT *r, XT *x, int a, int b) {
  if (!lines_pay(c, L)) {
    gs_block<VT, XT, ACC, ZA, FINE>(c, L, r, x, a);
    gs_block<VT, XT, ACC, ZB, FINE>(c, L, r, x, b);
    if constexpr (STEPS == 3) gs_block<VT, XT, ACC, -1, FINE>(c, L, r, x, a);
    return;
  }
  const int64_t ra = L.lay.start[a], rb = L.lay.start[b], nr = L.lay.start[a + 1] - ra;
  if (nr <= 0) return;  // a grid of one plane has no rows of an odd z
  const int line = L.lay.nx / 2, rows = line <= kSlice ? kSlice / line * line : line;
  const unsigned grid = (unsigned)((nr + rows - 1) / rows), bs = (unsigned)(rows + kSlice - 1) / kSlice * kSlice;
  const ColIdx cia = col_idx(c, L, a), cib = col_idx(c, L, b);
  with_forms<VT>(L, cia, [&](auto CF, auto VF) {
    if constexpr (CF() != kColsStored)
      k_gs_lines<VT, XT, ACC, ZA, ZB, STEPS, FINE, VF()>
          <<<grid, bs, 0, c->stream>>>(cia, cib, val_src<VT, ACC>(L), r, x, ra, rb, nr, rows);
  });
}

// Steps of blocks a, b, whose classes differ in z alone.
template <class VT, class XT, class ACC, int ZA, int ZB, bool FINE>
static void gs_columns(Ctx *c, const Level &L, const XT *r, XT *x, int a, int b) {
  if (!columns_pay(c, L)) {
    gs_block<VT, XT, ACC, ZA, FINE>(c, L, r, x, a);
    gs_block<VT, XT, ACC, ZB, FINE>(c, L, r, x, b);
    return;
  }
  const int64_t ra = L.lay.start[a], rb = L.lay.start[b], nr = L.lay.start[a + 1] - ra;
  if (nr <= 0) return;
  const int plane = L.lay.nx / 2 * (L.lay.ny / 2), nz = L.lay.nz / 2, cols = kBlock / nz;
  const unsigned grid = (unsigned)((plane + cols - 1) / cols) + (nr > (int64_t)plane * nz ? 1 : 0);
  const ColIdx cia = col_idx(c, L, a), cib = col_idx(c, L, b);
  with_forms<VT>(L, cia, [&](auto CF, auto VF) {
    if constexpr (CF() != kColsStored)
      k_gs_columns<VT, XT, ACC, ZA, ZB, FINE, VF()>
          <<<grid, kBlock, 0, c->stream>>>(cia, cib, val_src<VT, ACC>(L), r, x, ra, rb, nr, plane, nz, cols);
  });
}

// The zero-start forward sweep of the default order: block k reads only the
// blocks swept before it.  The backward step of block 6 comes with it.
template <class VT, class XT, class ACC, bool FINE>
static void zero_start_forward(Ctx *c, const Level &L, const XT *r, XT *x) {
  gs_columns<VT, XT, ACC, 0, 1, FINE>(c, L, r, x, 0, 1);
  gs_lines<VT, XT, ACC, 2, 3, 2, FINE>(c, L, r, x, 2, 3);
  gs_columns<VT, XT, ACC, 4, 5, FINE>(c, L, r, x, 4, 5);
  gs_lines<VT, XT, ACC, 6, 7, 3, FINE>(c, L, r, x, 6, 7);
}

// The remaining backward steps of the default order, from block 5.
template <class VT, class XT, class ACC, bool FINE>
static void backward_from_5(Ctx *c, const Level &L, const XT *r, XT *x) {
  gs_columns<VT, XT, ACC, -1, -1, FINE>(c, L, r, x, 5, 4);
  gs_lines<VT, XT, ACC, -1, -1, 2, FINE>(c, L, r, x, 3, 2);
  gs_columns<VT, XT, ACC, -1, -1, FINE>(c, L, r, x, 1, 0);
}

template <class XT>
__global__ __launch_bounds__(kBlock) void k_zero(XT *__restrict__ x, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i < n) x[i] = (XT)0;
}

static bool default_order(const Level &L) {
  if (L.lay.general) return false;
  for (int k = 0; k < kColours; ++k)
    if (L.lay.cls[k] != kDefaultOrder[k]) return false;
  return true;
}

// r.x partials of a level as its post-smoother's steps leave them (k_gs with
// RZ): the tiles of the last block, then of the blocks down to the first, each
// block's in the order of its launch.
struct RzBlocks {
  int start[kTailColours + 1];
  int ncol;
};
__global__ __launch_bounds__(kBlock) void k_rz(const RzBlocks L, const double *__restrict__ r,
                                               const double *__restrict__ x, double *rz) {
  int k = L.ncol - 1, first = 0, n = 0;
  for (;; --k) {
    n = (L.start[k + 1] - L.start[k] + kBlock - 1) / kBlock;
    if ((int)blockIdx.x < first + n) break;
    first += n;
  }
  const int64_t row = L.start[k] + tile_at<HPCGX_FINE_ROT != 0>((int)blockIdx.x - first, n) * kBlock + threadIdx.x;
  const double v[1] = {row < L.start[k + 1] ? r[row] * x[row] : 0.0};
  block_partials<1>(v, rz);
}
// Returns the number of partials.
static int64_t rz_pass(Ctx *c, const Level &L, const double *r, const double *x, double *rz) {
  RzBlocks b;
  b.ncol = L.lay.ncol;
  int64_t n = 0;
  for (int k = 0; k <= b.ncol; ++k) b.start[k] = (int)L.lay.start[k];
  for (int k = 0; k < b.ncol; ++k) n += tiles(b.start[k + 1] - b.start[k]);
  k_rz<<<(unsigned)n, kBlock, 0, c->stream>>>(b, r, x, rz);
  return n;
}

// One symmetric Gauss-Seidel step over the colour blocks.  Forward sweep
// blocks 0..ncol-1, backward sweep ncol-2..0: the backward step of the last
// block would recompute it from exactly the neighbour values its forward step
// used, so it is elided.  zero_start: x is known to be zero on entry (the
// V-cycle's first sweep); in the default stencil order x is then not read
// before it is written; otherwise (general levels, other orders) it is
// zero-filled first, and block 0, whose neighbours are all still zero, reads
// only its diagonal (x_i = r_i / a_ii, what the full step gives bit for bit).
// rz: the steps that leave their rows final (forward step of the last block,
// then the backward steps) write r.x partials at rz, *nrz of them in all.
// x may hold anything on a zero start (a caller's vector, or a coarse level's after
// a V-cycle on a non-finite input): see mend_nan.
template <class VT, class XT, class ACC, bool FINE>
static void sweep(Ctx *c, const Level &L, const XT *r, XT *x, bool zero_start, double *rz = nullptr,
                  int64_t *nrz = nullptr) {
  if (zero_start && !default_order(L)) {
    k_zero<XT><<<tiles(L.lay.npad), kBlock, 0, c->stream>>>(x, L.lay.npad);
    gs_block<VT, XT, ACC, 0, FINE>(c, L, r, x, 0);
    for (int k = 1; k < L.lay.ncol; ++k) gs_block<VT, XT, ACC, -1, FINE>(c, L, r, x, k);
  } else if (zero_start) {
    zero_start_forward<VT, XT, ACC, FINE>(c, L, r, x);
    backward_from_5<VT, XT, ACC, FINE>(c, L, r, x);
    return;
  } else if (default_order(L) && (!rz || lines_pay(c, L))) {
    gs_columns<VT, XT, ACC, -1, -1, FINE>(c, L, r, x, 0, 1);
    gs_lines<VT, XT, ACC, -1, -1, 2, FINE>(c, L, r, x, 2, 3);
    gs_columns<VT, XT, ACC, -1, -1, FINE>(c, L, r, x, 4, 5);
    gs_lines<VT, XT, ACC, -1, -1, 3, FINE>(c, L, r, x, 6, 7);
    backward_from_5<VT, XT, ACC, FINE>(c, L, r, x);
    // a pass of its own for r.x costs less than the launches that the pairs save
    if constexpr (sizeof(XT) == 8) {
      if (rz) *nrz = rz_pass(c, L, r, x, rz);
    }
    return;
  } else {
    for (int k = 0; k + 1 < L.lay.ncol; ++k) gs_block<VT, XT, ACC, -1, FINE>(c, L, r, x, k);
    const int last = L.lay.ncol - 1;
    gs_block<VT, XT, ACC, -1, FINE>(c, L, r, x, last, rz);
    if (rz) rz += tiles(L.lay.start[last + 1] - L.lay.start[last]);
  }
  for (int k = L.lay.ncol - 2; k >= 0; --k) {
    gs_block<VT, XT, ACC, -1, FINE>(c, L, r, x, k, rz);
    if (rz) rz += tiles(L.lay.start[k + 1] - L.lay.start[k]);
  }
  if (nrz) {
    *nrz = 0;
    for (int k = 0; k < L.lay.ncol; ++k) *nrz += tiles(L.lay.start[k + 1] - L.lay.start[k]);
  }
}

template <class VT, class XT, class ACC>
static int symgs_launch(Ctx *c, int l, const XT *r, XT *x, bool zero_start, double *rz = nullptr,
                        int64_t *nrz = nullptr) {
  const Level &L = c->levels[l];
  if (l == 0) sweep<VT, XT, ACC, true>(c, L, r, x, zero_start, rz, nrz);
  else sweep<VT, XT, ACC, false>(c, L, r, x, zero_start);
  HPCGX_CHECK_LAUNCH(c);
  return HPCGX_OK;
}

// Runs the V-cycle from level l down (or, with load_x, a smoothing step of
// level l alone) in one workgroup.  False: these levels take launches, being
// too large, of different forms, or of more colours than the kernel sweeps.
template <class VT, class XT, class ACC, bool SCALE>
static bool tail(Ctx *c, int l, const XT *r, XT *x, bool load_x = false) {
  const Level &F = c->levels[l];
  if (F.lay.npad > kTailRows) return false;
  TailArgs<VT, XT, ACC> a;
  a.r = r;
  a.x = x;
  a.n = load_x ? 1 : (int)c->levels.size() - l;
  a.load_x = load_x;
  const ColIdx ci = col_idx(c, F);
  int64_t off = 0;
  int waves = 1;
  for (int k = 0; k < a.n; ++k) {
    const Level &L = c->levels[l + k];
    TailLevel<VT, XT, ACC> &t = a.lv[k];
    t.ci = col_idx(c, L);
    if (L.lay.ncol > kTailColours || !L.dslot != !F.dslot || !t.ci.cbase != !ci.cbase ||
        val_form<VT>(L, t.ci) != val_form<VT>(F, ci) || (L.frow && !F.dslot))
      return false;
    t.src = val_src<VT, ACC>(L);
    t.dslot = L.dslot;
    t.inj = L.inj;
    t.frow = L.frow;
    t.sigma = L.sigma;
    t.boffs = L.diag_one ? L.boffs : nullptr;
    t.ninj = (int)L.ninj;
    t.row0 = (int)L.lay.start[L.lay.inj];
    t.npad = (int)L.lay.npad;
    t.ncol = L.lay.ncol;
    for (int j = 0; j <= L.lay.ncol; ++j) t.start[j] = (int)L.lay.start[j];
    int slices = 1;
    for (int j = 0; j < L.lay.ncol; ++j) slices = std::max(slices, (t.start[j + 1] - t.start[j]) >> 6);
    if (slices > kTailThreads / kSlice) t.boffs = nullptr;
    waves = std::max(waves, slices);
    t.xoff = (int)off;
    t.roff = (int)(off + L.lay.npad + 1);
    off += 2 * L.lay.npad + 1;
    if (off * (int64_t)sizeof(XT) > kTailLds) return false;
  }
  const unsigned lds = (unsigned)(off * sizeof(XT));
  const unsigned bs = (unsigned)std::min(waves, kTailThreads / kSlice) * kSlice;
  auto go = [&](auto CF, auto VF, auto GEN) {
    const auto kernel = k_tail<VT, XT, ACC, SCALE, CF(), VF(), GEN()>;
    static std::atomic<uint64_t> raised{0};  // devices on which the kernel may take all of a CU's LDS
    const uint64_t bit = (uint64_t)1 << (c->device & 63);
    if (!(raised.load() & bit)) {
      (void)hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, kTailLds);
      raised.fetch_or(bit);
    }
    kernel<<<1, bs, lds, c->stream>>>(a);
  };
  if (F.dslot) {
    constexpr std::integral_constant<int, kValsStored> stored{};
    if (ci.cbase) go(std::integral_constant<int, kColsSlice>{}, stored, std::true_type{});
    else go(std::integral_constant<int, kColsStored>{}, stored, std::true_type{});
  } else {
    // a kappa level reads its stored values here: the field's 27 gathers would
    // not come from LDS (20^3 fp64, 2 levels: 143 us against 93)
    with_forms<VT>(F, ci, [&](auto CF, auto VF) {
      go(CF, std::integral_constant<int, VF() == kValsSlot ? kValsSlot : kValsStored>{}, std::false_type{});
    });
  }
  return true;
}

// V-cycle of ComputeMG_ref.cpp:39-63: x = 0; pre-smooth; residual + restrict;
// recurse; prolong; post-smooth.  The coarsest level gets one smoothing step.
// rz / nrz: r.x partials of the result from the post-smoother (see sweep);
// from level 0 of an fp64 stencil hierarchy with a coarse level only.
template <class VT, class XT, class ACC, bool SCALE>
static int vcycle(Ctx *c, int l, const XT *r, XT *x, double *rz = nullptr, int64_t *nrz = nullptr) {
  const Level &L = c->levels[l];
  if (tail<VT, XT, ACC, SCALE>(c, l, r, x)) {
    if constexpr (sizeof(VT) == 8) {
      if (rz) *nrz = rz_pass(c, L, r, x, rz);
    }
    HPCGX_CHECK_LAUNCH(c);
    return HPCGX_OK;
  }
  int rc = symgs_launch<VT, XT, ACC>(c, l, r, x, true);
  if (rc || l + 1 >= (int)c->levels.size()) return rc;
  Level &C = c->levels[l + 1];
  XT *rc_v, *xc_v;
  if constexpr (sizeof(XT) == 8) {
    rc_v = reinterpret_cast<XT *>(C.r);
    xc_v = reinterpret_cast<XT *>(C.x);
  } else {
    rc_v = reinterpret_cast<XT *>(C.r32);
    xc_v = reinterpret_cast<XT *>(C.x32);
  }
  const int64_t nc = L.ninj, r0 = L.lay.start[L.lay.inj];
  const ColIdx ci = col_idx(c, L, L.frow ? -1 : L.lay.inj);
  with_forms<VT, true>(L, ci, [&](auto CF, auto VF) {
    if constexpr (VF() != kValsStored && sizeof(XT) == 8) {
      if (!L.frow && run_rows(L, nc)) {
        k_restrict_run<VF()><<<run_tiles(nc), kBlock, 0, c->stream>>>(ci, val_src<VT, ACC>(L), r, x, rc_v, L.inj, r0, nc);
        return;
      }
    }
    k_restrict<VT, XT, ACC, SCALE, CF(), VF()><<<tiles(nc), kBlock, 0, c->stream>>>(
        ci, val_src<VT, ACC>(L), r, x, rc_v, L.inj, L.sigma, r0, nc, L.frow);
  });
  HPCGX_CHECK_LAUNCH(c);
  if ((rc = vcycle<VT, XT, ACC, SCALE>(c, l + 1, rc_v, xc_v))) return rc;
  k_prolong<XT, ACC, SCALE><<<tiles(nc), kBlock, 0, c->stream>>>(x, xc_v, L.inj, L.sigma, r0, nc, L.frow);
  HPCGX_CHECK_LAUNCH(c);
  return symgs_launch<VT, XT, ACC>(c, l, r, x, false, rz, nrz);
}

// vector kernels

__global__ __launch_bounds__(kBlock) void k_waxpby(int64_t n, double alpha,
                                                   const double *__restrict__ x, double beta,
                                                   const double *__restrict__ y,
                                                   double *__restrict__ w) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  w[i] = waxpby1(alpha, x[i], beta, y[i]);
}

// out = x . y (ComputeDotProduct_ref.cpp:54-64, fixed-order tree)
__global__ __launch_bounds__(kBlock) void k_dot(int64_t n, const double *__restrict__ x,
                                                const double *__restrict__ y, double *partials) {
  double a[kChunk], b[kChunk];
#pragma unroll
  for (int j = 0; j < kChunk; ++j) {
    const int64_t i = chunk_index(j);
    a[j] = i < n ? x[i] : 0.0;
    b[j] = i < n ? y[i] : 0.0;
  }
  double acc = 0.0;
#pragma unroll
  for (int j = 0; j < kChunk; ++j) acc += a[j] * b[j];
  const double v[1] = {acc};
  block_partials<1>(v, partials);
}

// w = alpha x + beta y ; out = w . w   (WAXPBY then DOT of CG.cpp:88-89 / 122-123)
__global__ __launch_bounds__(kBlock) void k_waxpby_dot(int64_t n, double alpha,
                                                       const double *__restrict__ x, double beta,
                                                       const double *__restrict__ y,
                                                       double *__restrict__ w, double *partials) {
  double a[kChunk], b[kChunk];
#pragma unroll
  for (int j = 0; j < kChunk; ++j) {
    const int64_t i = chunk_index(j);
    a[j] = i < n ? x[i] : 0.0;
    b[j] = i < n ? y[i] : 0.0;
  }
  double acc = 0.0;
#pragma unroll
  for (int j = 0; j < kChunk; ++j) {
    const int64_t i = chunk_index(j);
    const double v = waxpby1(alpha, a[j], beta, b[j]);
    if (i < n) {
      w[i] = v;
      acc += v * v;
    }
  }
  const double v[1] = {acc};
  block_partials<1>(v, partials);
}


int mg_fp64(Ctx *c, int level, const double *r, double *x, double *rz, int64_t *nrz) {
  if (rz && (level + 1 >= (int)c->levels.size() || c->levels[level].lay.general))
    return set_err(c, HPCGX_EINVAL, "fused r.z needs a stencil level with a coarse level");
  return vcycle<double, double, double, false>(c, level, r, x, rz, nrz);
}

int mg_fp32(Ctx *c, int level, const float *r, float *x) {
  return vcycle<float, float, float, false>(c, level, r, x);
}

int zero_vec(Ctx *c, double *x, int64_t n) {
  k_zero<double><<<tiles(n), kBlock, 0, c->stream>>>(x, n);
  HPCGX_CHECK_LAUNCH(c);
  return HPCGX_OK;
}

int zero_vec(Ctx *c, float *x, int64_t n) {
  k_zero<float><<<tiles(n), kBlock, 0, c->stream>>>(x, n);
  HPCGX_CHECK_LAUNCH(c);
  return HPCGX_OK;
}

__global__ __launch_bounds__(kBlock) void k_scale(const float *__restrict__ a, const float *__restrict__ s,
                                                  float *__restrict__ o, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i < n) o[i] = a[i] * s[i];
}

// The scaled fp16 V-cycle proper: xhat from rhat = dinv r (a solver that
// applies the scalings itself).
int mg_fp16_scaled(Ctx *c, const float *rhat, float *xhat) {
  return vcycle<__half, float, float, true>(c, 0, rhat, xhat);
}

// Scaled fp16 V-cycle on level 0: rhat = dinv r, V-cycle with D^-1/2 A D^-1/2,
// x = dinv xhat.
int mg_fp16(Ctx *c, const float *r, float *x) {
  Level &L = c->levels[0];
  const int64_t np = L.lay.npad;
  k_scale<<<tiles(np), kBlock, 0, c->stream>>>(r, L.dinv, L.r16, np);
  HPCGX_CHECK_LAUNCH(c);
  int rc = vcycle<__half, float, float, true>(c, 0, L.r16, x);
  if (rc) return rc;
  k_scale<<<tiles(np), kBlock, 0, c->stream>>>(x, L.dinv, x, np);
  HPCGX_CHECK_LAUNCH(c);
  return HPCGX_OK;
}

__global__ __launch_bounds__(kBlock) void k_to_single(const double *__restrict__ a, float *__restrict__ o,
                                                      int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i < n) o[i] = (float)a[i];
}

__global__ __launch_bounds__(kBlock) void k_to_double(const float *__restrict__ a, double *__restrict__ o,
                                                      int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i < n) o[i] = (double)a[i];
}

int spmv_fp64(Ctx *c, int level, const double *x, double *y) {
  const Level &L = c->levels[level];
  const ColIdx ci = col_idx(c, L);
  with_forms<double>(L, ci, [&](auto CF, auto VF) {
    if constexpr (VF() != kValsStored) {
      if (run_rows(L, L.lay.npad)) {
        k_spmv_run<VF()><<<run_tiles(L.lay.npad), kBlock, 0, c->stream>>>(ci, val_src<double, double>(L), x, y, L.lay.npad,
                                                                       block_tiles(L));
        return;
      }
    }
    k_spmv<double, double, double, CF(), VF()><<<tiles(L.lay.npad), kBlock, 0, c->stream>>>(
        ci, val_src<double, double>(L), x, y, L.lay.npad);
  });
  HPCGX_CHECK_LAUNCH(c);
  return HPCGX_OK;
}

int symgs_fp64(Ctx *c, int level, const double *r, double *x) {
  if (tail<double, double, double, false>(c, level, r, x, true)) {
    HPCGX_CHECK_LAUNCH(c);
    return HPCGX_OK;
  }
  return symgs_launch<double, double, double>(c, level, r, x, false);
}

// ---------------------------------------------------------------------------
// Static scratch of hpcgx_dot_noalloc, the dot product for callers that may
// not allocate device memory.  It holds the partial sums of the producer
// blocks of a level of up to kNoAllocRows padded rows (one per 1024 rows),
// their folded sums and the finishing kernel's scalars: 2.1 MB, which each
// device keeps until the process ends.  Every call on one device shares it.
// Each call overwrites all it reads (every producer block writes its
// partial, the fold every folded sum, the finishing kernel the result), so
// nothing needs clearing.
constexpr int64_t kNoAllocRows = (int64_t)1 << 28;
constexpr int64_t kNaBlocks = kNoAllocRows / (kChunk * kBlock);
constexpr int64_t kNaFolded = kNaBlocks;                                    // offset of the folded sums
constexpr int64_t kNaScal = kNaFolded + (kNaBlocks / kFold + 1 + 31) / 32 * 32;  // offset of the scalars
constexpr int64_t kNaDoubles = kNaScal + S_COUNT;
static_assert(chunk_blocks(kNoAllocRows) == kNaBlocks, "one partial per producer block");
static __device__ __align__(256) double scratch[kNaDoubles];

// The device address of `scratch` on each device (the array's name is only a
// host-side handle), looked up once per device by noalloc_scratch_init.
constexpr int kNaDevices = 64;
static double *g_scratch[kNaDevices] = {};
static std::mutex g_scratch_mu;

int noalloc_scratch_init(int device) {
  if (device < 0 || device >= kNaDevices) return HPCGX_OK;  // the entry point refuses such devices
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (g_scratch[device]) return HPCGX_OK;
  void *p = nullptr;
  if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) return HPCGX_EHIP;
  g_scratch[device] = static_cast<double *>(p);
  return HPCGX_OK;
}

static double *noalloc_scratch(int device) {
  if (device < 0 || device >= kNaDevices) return nullptr;
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  return g_scratch[device];
}

}  // namespace hpcgx

using namespace hpcgx;

static int check_level(hpcgx_ctx *c, int level, const char *who) {
  if (!c) return HPCGX_EINVAL;
  if (level < 0 || level >= (int)c->levels.size())
    return set_err(c, HPCGX_EINVAL, std::string(who) + ": no such level");
  if (hipSetDevice(c->device) != hipSuccess) return set_err(c, HPCGX_EHIP, "hipSetDevice failed");
  return ensure_ready(c);
}

// Null pointers and vectors of the wrong size (those made by hpcgx_vec_alloc)
// are refused before any launch.
static int check_vecs(hpcgx_ctx *c, int64_t elems, const char *who, std::initializer_list<const void *> vs) {
  for (const void *v : vs) {
    if (!v) return set_err(c, HPCGX_EINVAL, std::string(who) + ": null vector");
    int rc = check_vec(c, v, elems, who);
    if (rc) return rc;
  }
  return HPCGX_OK;
}

static int64_t npad_of(hpcgx_ctx *c, int level) { return c->levels[level].lay.npad; }

extern "C" {

int hpcgx_spmv(hpcgx_ctx *c, int level, const double *x, double *y) {
  int rc = check_level(c, level, "spmv");
  if (rc) return rc;
  if ((rc = check_vecs(c, npad_of(c, level), "spmv", {x, y}))) return rc;
  if (x == y) return set_err(c, HPCGX_EINVAL, "spmv: x and y must be distinct device vectors");
  return spmv_fp64(c, level, x, y);
}

int hpcgx_symgs(hpcgx_ctx *c, int level, const double *r, double *x) {
  int rc = check_level(c, level, "symgs");
  if (rc) return rc;
  if ((rc = check_vecs(c, npad_of(c, level), "symgs", {r, x}))) return rc;
  return symgs_fp64(c, level, r, x);
}

int hpcgx_restrict(hpcgx_ctx *c, int level, const double *r, const double *x, double *rc_out) {
  int rc = check_level(c, level, "restrict");
  if (rc) return rc;
  if (level + 1 >= (int)c->levels.size()) return set_err(c, HPCGX_EINVAL, "restrict: level has no coarse level");
  if ((rc = check_vecs(c, npad_of(c, level), "restrict", {r, x})) ||
      (rc = check_vecs(c, npad_of(c, level + 1), "restrict", {rc_out})))
    return rc;
  const Level &L = c->levels[level];
  const int64_t nc = L.ninj;
  const ColIdx ci = col_idx(c, L, L.frow ? -1 : L.lay.inj);
  with_forms<double, true>(L, ci, [&](auto CF, auto VF) {
    if constexpr (VF() != kValsStored) {
      if (!L.frow && run_rows(L, nc)) {
        k_restrict_run<VF()><<<run_tiles(nc), kBlock, 0, c->stream>>>(ci, val_src<double, double>(L), r, x, rc_out, L.inj,
                                                                      L.lay.start[L.lay.inj], nc);
        return;
      }
    }
    k_restrict<double, double, double, false, CF(), VF()><<<tiles(nc), kBlock, 0, c->stream>>>(
        ci, val_src<double, double>(L), r, x, rc_out, L.inj, nullptr, L.lay.start[L.lay.inj], nc, L.frow);
  });
  HPCGX_CHECK_LAUNCH(c);
  return HPCGX_OK;
}

int hpcgx_prolong(hpcgx_ctx *c, int level, const double *xc, double *x) {
  int rc = check_level(c, level, "prolong");
  if (rc) return rc;
  if (level + 1 >= (int)c->levels.size()) return set_err(c, HPCGX_EINVAL, "prolong: level has no coarse level");
  if ((rc = check_vecs(c, npad_of(c, level + 1), "prolong", {xc})) ||
      (rc = check_vecs(c, npad_of(c, level), "prolong", {x})))
    return rc;
  const Level &L = c->levels[level];
  const int64_t nc = L.ninj;
  k_prolong<double, double, false><<<tiles(nc), kBlock, 0, c->stream>>>(x, xc, L.inj, nullptr,
                                                                        L.lay.start[L.lay.inj], nc, L.frow);
  HPCGX_CHECK_LAUNCH(c);
  return HPCGX_OK;
}

int hpcgx_mg(hpcgx_ctx *c, int level, const double *r, double *x) {
  int rc = check_level(c, level, "mg");
  if (rc) return rc;
  if ((rc = check_vecs(c, npad_of(c, level), "mg", {r, x}))) return rc;
  if (r == x) return set_err(c, HPCGX_EINVAL, "mg: r and x must be distinct device vectors");
  return mg_fp64(c, level, r, x);
}

int hpcgx_mg_mixed(hpcgx_ctx *c, int precision, const double *r, double *x) {
  int rc = check_level(c, 0, "mg_mixed");
  if (rc) return rc;
  if ((rc = check_vecs(c, npad_of(c, 0), "mg_mixed", {r, x}))) return rc;
  if (r == x) return set_err(c, HPCGX_EINVAL, "mg_mixed: r and x must be distinct device vectors");
  const int need = precision == HPCGX_PREC_FP32 ? 1 : precision == HPCGX_PREC_FP16 ? 2 : 0;
  if (!need) return set_err(c, HPCGX_EINVAL, "mg_mixed: precision must be HPCGX_PREC_FP32 or HPCGX_PREC_FP16");
  if (!(c->prepared & need)) return set_err(c, HPCGX_ESTATE, "mg_mixed: call hpcgx_prepare_precision first");
  const int64_t np = c->levels[0].lay.npad;
  k_to_single<<<tiles(np), kBlock, 0, c->stream>>>(r, c->cg_r32, np);
  HPCGX_CHECK_LAUNCH(c);
  rc = precision == HPCGX_PREC_FP32 ? mg_fp32(c, 0, c->cg_r32, c->cg_z32)
                                    : mg_fp16(c, c->cg_r32, c->cg_z32);
  if (rc) return rc;
  k_to_double<<<tiles(np), kBlock, 0, c->stream>>>(c->cg_z32, x, np);
  HPCGX_CHECK_LAUNCH(c);
  return HPCGX_OK;
}

// The vector hooks take the reference's n = nrow (ComputeDotProduct.cpp:41,
// ComputeWAXPBY.cpp:42: the whole level-0 vector).  Device vectors are in
// colour order, where the first k entries are not the first k natural rows,
// so any other length has no reference meaning and is refused; npad (the
// padded length, padding entries zero) is accepted as the same vector.
static int check_n(hpcgx_ctx *c, int64_t n, const char *who) {
  int rc = check_level(c, 0, who);
  if (rc) return rc;
  const Layout &lay = c->levels[0].lay;
  if (n != lay.n && n != lay.npad)
    return set_err(c, HPCGX_EINVAL, std::string(who) + ": n must be the level-0 row count (" +
                                        std::to_string((long long)lay.n) + ")");
  return HPCGX_OK;
}

// n = the level's row count covers the whole padded vector.
static int64_t span(hpcgx_ctx *c, int64_t) { return c->levels[0].lay.npad; }

int hpcgx_dot(hpcgx_ctx *c, int64_t n, const double *x, const double *y, double *result) {
  int rc = check_n(c, n, "dot");
  if (rc) return rc;
  if (!result) return set_err(c, HPCGX_EINVAL, "dot: null argument");
  const int64_t m = span(c, n);
  if ((rc = check_vecs(c, m, "dot", {x, y}))) return rc;
  k_dot<<<chunk_blocks(m), kBlock, 0, c->stream>>>(m, x, y, c->partials);
  HPCGX_CHECK_LAUNCH(c);
  if ((rc = finish(c, 1, chunk_blocks(m), F_DOT, nullptr, c->hsum))) return rc;
  return wait_host(c, c->hsum, result);
}

int hpcgx_waxpby(hpcgx_ctx *c, int64_t n, double alpha, const double *x, double beta, const double *y,
                 double *w) {
  int rc = check_n(c, n, "waxpby");
  if (rc) return rc;
  const int64_t m = span(c, n);
  if ((rc = check_vecs(c, m, "waxpby", {x, y, w}))) return rc;
  k_waxpby<<<tiles(m), kBlock, 0, c->stream>>>(m, alpha, x, beta, y, w);
  HPCGX_CHECK_LAUNCH(c);
  return HPCGX_OK;
}

int hpcgx_waxpby_dot(hpcgx_ctx *c, int64_t n, double alpha, const double *x, double beta, const double *y,
                     double *w, double *result) {
  int rc = check_n(c, n, "waxpby_dot");
  if (rc) return rc;
  if (!result) return set_err(c, HPCGX_EINVAL, "waxpby_dot: null argument");
  const int64_t m = span(c, n);
  if ((rc = check_vecs(c, m, "waxpby_dot", {x, y, w}))) return rc;
  k_waxpby_dot<<<chunk_blocks(m), kBlock, 0, c->stream>>>(m, alpha, x, beta, y, w, c->partials);
  HPCGX_CHECK_LAUNCH(c);
  if ((rc = finish(c, 1, chunk_blocks(m), F_DOT, nullptr, c->hsum))) return rc;
  return wait_host(c, c->hsum, result);
}

// hpcgx_dot with its partial sums in the static scratch instead of the
// context's buffers: the same kernels in the same order, so the same bits.
// Allocates nothing; the problem must already be set up (the context ready).
int hpcgx_dot_noalloc(hpcgx_ctx *c, int64_t n, const double *x, const double *y, double *result) {
  if (!c) return HPCGX_EINVAL;
  if (c->levels.empty() || !c->ready)
    return set_err(c, HPCGX_ESTATE, "dot_noalloc: no problem set up (it allocates nothing, so it cannot set one up)");
  if (!result) return set_err(c, HPCGX_EINVAL, "dot_noalloc: null argument");
  if (hipSetDevice(c->device) != hipSuccess) return set_err(c, HPCGX_EHIP, "hipSetDevice failed");
  const Layout &lay = c->levels[0].lay;
  if (n != lay.n && n != lay.npad)
    return set_err(c, HPCGX_EINVAL, "dot_noalloc: n must be the level-0 row count (" +
                                        std::to_string((long long)lay.n) + ")");
  const int64_t m = lay.npad;
  if (m > kNoAllocRows)
    return set_err(c, HPCGX_EINVAL, "dot_noalloc: the level has " + std::to_string((long long)m) +
                                        " padded rows; its static scratch covers at most 2^28 (use hpcgx_dot)");
  double *s = noalloc_scratch(c->device);
  if (!s) return set_err(c, HPCGX_ESTATE, "dot_noalloc: no static scratch on this device");
  int rc = check_vecs(c, m, "dot_noalloc", {x, y});
  if (rc) return rc;
  int64_t grid = chunk_blocks(m);
  k_dot<<<(unsigned)grid, kBlock, 0, c->stream>>>(m, x, y, s);
  HPCGX_CHECK_LAUNCH(c);
  const double *src = s;
  if (grid > kFoldAbove) {
    const int64_t g2 = (grid + kFold - 1) / kFold;
    k_fold<1><<<(unsigned)g2, kBlock, 0, c->stream>>>(s, grid, s + kNaFolded);
    src = s + kNaFolded;
    grid = g2;
  }
  k_finish<1><<<1, kFinishThreads, 0, c->stream>>>(src, grid, s + kNaScal, F_DOT, nullptr, c->hbuf);
  HPCGX_CHECK_LAUNCH(c);
  HPCGX_HIP(c, hipStreamSynchronize(c->stream));
  *result = c->hbuf[0];
  return HPCGX_OK;
}

}  // extern "C"
