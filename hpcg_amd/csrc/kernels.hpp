// Device kernels of the PCG iteration phase (gfx950, wave64).
//
// Matrix storage: 27-slot sliced ELL.  Slot s of a row is the stencil offset
// (dx,dy,dz) = (s%3-1, s/3%3-1, s/9-1); a neighbour outside the grid is a
// zero value whose explicit column is the row itself.  Within a slice of 64
// rows one wavefront reads the fp64 values of a pair of slots of its 64 rows
// as one contiguous 1024-byte run, 16 bytes per lane (the fp32 and fp16
// copies: four slots per load; val_pos), and each slot's column as a
// 256-byte run of explicit indices, a 64-byte run of int8 deltas, or no
// per-entry index at all (ColForm).  Rows are summed in slot
// order, ascending column order, the order in which the reference sums a row
// (ComputeSPMV_ref.cpp:67-68); the zero slots add exact zeros, so sums match
// the reference bit for bit.  The whole library is compiled with
// -ffp-contract=off: products and sums are rounded separately, as in the
// reference's x86-64 build.
#pragma once

#include <type_traits>
#include <utility>

#include "common.hpp"

namespace hpcgx {

__device__ __forceinline__ size_t ell_base(int64_t row) {
  return (size_t)(row >> 6) * (kSlots * kSlice) + (size_t)(row & 63);
}

// Blocks are dealt round-robin to the 8 XCDs; remap so that each XCD works on
// one contiguous range of tiles and neighbouring rows share that XCD's L2.
// ROT (the fine level's fp64 Gauss-Seidel steps): XCD x starts its range at
// x/8 of it and wraps.  A step's 8 ranges are slabs of one colour block,
// equally spaced in memory, and swept in lockstep they meet the same HBM
// channels at the same time; rotated, the fine 192^3 step took 57.6 us
// instead of 59.3 (explicit indices, one value slot per load; 4 alternating
// processes each).  Whole-level passes (SpMV)
// keep the plain map: there XCD x sweeps block x, and in lockstep the 8 XCDs
// gather x around the same grid position, which the last-level cache serves
// once (rotated, the 512^3 SpMV took 9.2-9.6 ms instead of 8.1-8.5).  The
// fp32 / fp16 steps keep it too (rotated, the mixed 512^3 solves ran 1.7 %
// slower).
template <bool ROT = false>
__device__ __forceinline__ int64_t tile_at(int64_t b, int64_t G) {
  const int64_t per = G >> 3, rem = G & 7, xcd = b & 7, idx = b >> 3;
  int64_t r = idx;
  if constexpr (ROT) {
    const int64_t len = per + (xcd < rem ? 1 : 0);
    r += (xcd * len) >> 3;
    if (r >= len) r -= len;
  }
  return xcd * per + (xcd < rem ? xcd : rem) + r;
}
template <bool ROT = false>
__device__ __forceinline__ int64_t tile_id() {
  return tile_at<ROT>(blockIdx.x, gridDim.x);
}

// Tile of a whole-level pass that takes the 8 colour blocks together: XCD x
// gets the x-th eighth of every block, the blocks in turn, so one XCD's L2
// serves the 8 tiles that gather the same part of the vector.  bt: tiles per
// block, a multiple of 8 (block_tiles), or 0 for tile_id.
__device__ __forceinline__ int64_t level_tile(int bt) {
  if (!bt) return tile_id();
  const int xcd = blockIdx.x & 7, i = blockIdx.x >> 3;
  return (int64_t)(i & 7) * bt + xcd * (bt >> 3) + (i >> 3);
}

// The block index b with tile_id<ROT>() == tile in a grid of G blocks: where
// the one-row-per-lane launch of a pass leaves that tile's partial sum.
template <bool ROT = false>
__device__ __forceinline__ int64_t tile_slot(unsigned tile, unsigned G) {
  const unsigned per = G >> 3, rem = G & 7, wide = rem * (per + 1);
  unsigned xcd, r;
  if (tile < wide) {
    xcd = tile / (per + 1);
    r = tile - xcd * (per + 1);
  } else {
    xcd = rem + (tile - wide) / per;
    r = tile - wide - (xcd - rem) * per;
  }
  if constexpr (ROT) {
    const unsigned len = per + (xcd < rem ? 1 : 0), shift = (xcd * len) >> 3;
    r = r >= shift ? r - shift : r + len - shift;
  }
  return (int64_t)r * 8 + xcd;
}

// Where a launch takes its columns from.
enum ColSource : int {
  kColsStored = 0,  // the explicit 32-bit index of every entry
  kColsSlice = 1,   // the compact form: the slice's record, and its deltas (ColForm)
  kColsBlock = 2,   // the column is the row plus a distance that the slot has over the whole colour block
};

// Occupancy of the fp64 sparse kernels (SpMV, Gauss-Seidel steps,
// restriction).  With explicit 32-bit column indices: at most two waves per
// SIMD, so a wave holds the column, value and gather loads of all its slots
// in flight instead of the default's batches of about 9 at six waves per
// SIMD (measured with one value slot per load: 3 % faster at 512^3, the CG
// SpMV 9 %, 1.7 % at 192^3; eight waves per SIMD was 10 % slower; with
// paired values the explicit-column 192^3 set ran 1058 GFLOP/s at two, 1047
// at four and 1022 at eight, the general 128^3 layout 776, 779 and 670;
// HPCGX_FP64_WAVES overrides it at build time).  With
// compact columns (the default) a uniform slice needs no index load, all
// loads of a row still issue before the first wait (114 VGPRs for the fine
// step with paired values), and no limit is best: measured in alternating
// processes with one value slot per load, the 192^3 sets ran 1245-1249
// GFLOP/s unlimited, 1248-1249 at four waves per SIMD, 1241 at three and
// 1181 at two; the 512^3 FP64 solve 37.9-38.3 ms per iteration unlimited
// against 40.7-41.5 at two.  HPCGX_CI_FP64_WAVES overrides it at build time.  The
// fp32 / fp16 kernels keep the default, and so do steps that read fewer
// than 8 slots (the backend pads every kernel under the limit to its
// register budget).
#ifndef HPCGX_CI_FP64_WAVES
#define HPCGX_CI_FP64_WAVES 8
#endif
#ifndef HPCGX_FP64_WAVES
#define HPCGX_FP64_WAVES 2
#endif
template <class VT, int CF = kColsStored, int SLOTS = 27>
struct SparseOccupancy {
  static constexpr unsigned max_waves =
      (sizeof(VT) == 8 && SLOTS >= 8) ? (CF ? HPCGX_CI_FP64_WAVES : HPCGX_FP64_WAVES) : 8;
};
#define HPCGX_SPARSE_OCCUPANCY(VT, CF) __attribute__((amdgpu_waves_per_eu(1, SparseOccupancy<VT, CF>::max_waves)))

// Matrix loads.  NT (non-temporal): the fine level's matrix is streamed once
// per pass and is far larger than any cache, so it is kept out of the way of
// the vectors; coarse-level matrices fit in the 256 MB Infinity Cache and
// are loaded normally so that the V-cycle's repeated passes can hit there.
template <bool NT = true>
__device__ __forceinline__ int ld_col(const int *p) {
  if constexpr (NT) return __builtin_nontemporal_load(p);
  else return *p;
}
template <class ACC, bool NT = true>
__device__ __forceinline__ ACC ld_val(const double *p) {
  if constexpr (NT) return (ACC)__builtin_nontemporal_load(p);
  else return (ACC)*p;
}
template <class ACC, bool NT = true>
__device__ __forceinline__ ACC ld_val(const float *p) {
  if constexpr (NT) return (ACC)__builtin_nontemporal_load(p);
  else return (ACC)*p;
}
template <class ACC, bool NT = true>
__device__ __forceinline__ ACC ld_val(const __half *p) {
  const unsigned short *q = reinterpret_cast<const unsigned short *>(p);
  unsigned short bits;
  if constexpr (NT) bits = __builtin_nontemporal_load(q);
  else bits = *q;
  return (ACC)__half2float(__ushort_as_half(bits));
}

// The values of a unit of a row (val_pos): 2 or 4 adjacent values read with
// one load per lane -- a pair of fp64 values in 16 bytes, a quad of fp32 in
// 16, a quad of fp16 in 8, a pair of fp32 or fp16 in 8 or 4.
typedef double f64x2_t __attribute__((ext_vector_type(2)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef unsigned u32x2_t __attribute__((ext_vector_type(2)));
template <class V, bool NT>
__device__ __forceinline__ V ld_vec(const V *q) {
  if constexpr (NT) return __builtin_nontemporal_load(q);
  else return *q;
}
template <class ACC>
__device__ __forceinline__ ACC half_lo(unsigned bits) {
  return (ACC)__half2float(__ushort_as_half((unsigned short)(bits & 0xffffu)));
}
template <class ACC>
__device__ __forceinline__ ACC half_hi(unsigned bits) {
  return (ACC)__half2float(__ushort_as_half((unsigned short)(bits >> 16)));
}
template <class ACC, bool NT>
__device__ __forceinline__ void ld_unit(const double *p, ACC *a, std::integral_constant<int, 2>) {
  const f64x2_t v = ld_vec<f64x2_t, NT>(reinterpret_cast<const f64x2_t *>(p));
  a[0] = (ACC)v.x;
  a[1] = (ACC)v.y;
}
template <class ACC, bool NT>
__device__ __forceinline__ void ld_unit(const float *p, ACC *a, std::integral_constant<int, 2>) {
  const f32x2_t v = ld_vec<f32x2_t, NT>(reinterpret_cast<const f32x2_t *>(p));
  a[0] = (ACC)v.x;
  a[1] = (ACC)v.y;
}
template <class ACC, bool NT>
__device__ __forceinline__ void ld_unit(const float *p, ACC *a, std::integral_constant<int, 4>) {
  const f32x4_t v = ld_vec<f32x4_t, NT>(reinterpret_cast<const f32x4_t *>(p));
  a[0] = (ACC)v.x;
  a[1] = (ACC)v.y;
  a[2] = (ACC)v.z;
  a[3] = (ACC)v.w;
}
template <class ACC, bool NT>
__device__ __forceinline__ void ld_unit(const __half *p, ACC *a, std::integral_constant<int, 2>) {
  const unsigned bits = ld_vec<unsigned, NT>(reinterpret_cast<const unsigned *>(p));
  a[0] = half_lo<ACC>(bits);
  a[1] = half_hi<ACC>(bits);
}
template <class ACC, bool NT>
__device__ __forceinline__ void ld_unit(const __half *p, ACC *a, std::integral_constant<int, 4>) {
  const u32x2_t bits = ld_vec<u32x2_t, NT>(reinterpret_cast<const u32x2_t *>(p));
  a[0] = half_lo<ACC>(bits.x);
  a[1] = half_hi<ACC>(bits.x);
  a[2] = half_lo<ACC>(bits.y);
  a[3] = half_hi<ACC>(bits.y);
}

template <class F, int... U>
__device__ __forceinline__ void for_each_unit(F &&f, std::integer_sequence<int, U...>) {
  (f(std::integral_constant<int, U>{}), ...);
}

// Slots of a unit as a mask.
__host__ __device__ constexpr uint32_t unit_mask(const ValUnit &w) {
  uint32_t m = 0;
  for (int h = 0; h < w.n; ++h) m |= 1u << w.s[h];
  return m;
}

// The values of the slots in MASK of a row, into v[slot]; other entries of v
// are left unset.  A unit is read whole when any of its slots is wanted.
constexpr uint32_t kAllSlots = (1u << kSlots) - 1;
template <class ACC, bool NT, uint32_t MASK, class VT>
__device__ __forceinline__ void row_vals(const VT *__restrict__ vals, int64_t row, ACC (&v)[kSlots]) {
  constexpr int W = val_width<VT>;
  const VT *sb = vals + (size_t)(row >> 6) * (kSlots * kSlice);
  const int lane = (int)(row & 63);
  for_each_unit(
      [&](auto uc) {
        constexpr int u = decltype(uc)::value;
        constexpr ValUnit w = val_unit(W, u);
        constexpr int off = val_unit_off(W, u);
        if constexpr ((MASK & unit_mask(w)) != 0) {
          if constexpr (w.n == 1) {
            v[w.s[0]] = ld_val<ACC, NT>(sb + off + lane);
          } else {
            ACC t[w.n];
            ld_unit<ACC, NT>(sb + off + w.n * lane, t, std::integral_constant<int, w.n>{});
#pragma unroll
            for (int h = 0; h < w.n; ++h) v[w.s[h]] = t[h];
          }
        }
      },
      std::make_integer_sequence<int, val_units(W)>{});
}

// A launch's value source: the stored values, the row masks, the slot values
// (kValsSlot) and the field (kValsField).
template <class VT, class ACC>
struct ValSrc {
  const VT *vals;
  const uint32_t *mask;
  const ACC *slotv;
  const double *field;
  int diag_one;  // kValsSlot: the diagonal is slotv[13] on every row
};

// v where bit s of m is set, else +0: two or three integer operations, no
// branch and no compare.
__device__ __forceinline__ double bit_select(uint32_t m, int s, double v) {
  const int k = (int)(m << (31 - s)) >> 31;
  return __hiloint2double(__double2hiint(v) & k, __double2loint(v) & k);
}
__device__ __forceinline__ float bit_select(uint32_t m, int s, float v) {
  const int k = (int)(m << (31 - s)) >> 31;
  return __int_as_float(__float_as_int(v) & k);
}

// The off-diagonal values of one row in any form.  load() issues the row's
// loads; at(s, c) is the value of slot s, whose column is c.
template <int VF, class VT, class ACC, bool NT, uint32_t MASK>
struct RowVals;

template <class VT, class ACC, bool NT, uint32_t MASK>
struct RowVals<kValsStored, VT, ACC, NT, MASK> {
  ACC v[kSlots];
  __device__ __forceinline__ void load(const ValSrc<VT, ACC> &src, int64_t row) {
    row_vals<ACC, NT, MASK>(src.vals, row, v);
  }
  __device__ __forceinline__ ACC at(int s, int) const { return v[s]; }
  // the diagonal of a stencil row
  __device__ __forceinline__ ACC diag(const ValSrc<VT, ACC> &src, int64_t row) const {
    if constexpr ((MASK >> kDiagSlot) & 1u) return v[kDiagSlot];
    else return ld_val<ACC, NT>(src.vals + val_pos<val_width<VT>>(row, kDiagSlot));
  }
};

template <class VT, class ACC, bool NT, uint32_t MASK>
struct RowVals<kValsSlot, VT, ACC, NT, MASK> {
  uint32_t m;
  ACC d;
  const ACC *slotv;
  __device__ __forceinline__ void load(const ValSrc<VT, ACC> &src, int64_t row) {
    slotv = src.slotv;
    if constexpr (NT) m = __builtin_nontemporal_load(src.mask + row);
    else m = src.mask[row];
    if (src.diag_one) d = (m >> kDiagSlot) & 1u ? slotv[kDiagSlot] : (ACC)1;  // padding: the identity row
    else d = ld_val<ACC, NT>(src.vals + val_pos<val_width<VT>>(row, kDiagSlot));
  }
  __device__ __forceinline__ ACC at(int s, int) const { return s == kDiagSlot ? d : bit_select(m, s, slotv[s]); }
  __device__ __forceinline__ ACC diag(const ValSrc<VT, ACC> &, int64_t) const { return d; }
};

template <class VT, class ACC, bool NT, uint32_t MASK>
struct RowVals<kValsField, VT, ACC, NT, MASK> {
  uint32_t m;
  ACC d;
  double ki;
  const double *field;
  __device__ __forceinline__ void load(const ValSrc<VT, ACC> &src, int64_t row) {
    field = src.field;
    if constexpr (NT) m = __builtin_nontemporal_load(src.mask + row);
    else m = src.mask[row];
    ki = field[row];
    d = ld_val<ACC, NT>(src.vals + val_pos<val_width<VT>>(row, kDiagSlot));
  }
  __device__ __forceinline__ ACC at(int s, int c) const {
    return s == kDiagSlot ? d : bit_select(m, s, (ACC)(-((ki + field[c]) * 0.5)));
  }
  __device__ __forceinline__ ACC diag(const ValSrc<VT, ACC> &, int64_t) const { return d; }
};

// Column index of (row, slot): the explicit 32-bit index, the compact form
// (ColForm) with a per-slice base, or, in a launch over rows of one colour
// block, the row plus the slot's distance.
struct ColIdx {
  const int *cols;
  const int *cbase;     // null: explicit indices only
  const int8_t *cdelta;
  const uint8_t *cform;
  const int *off;   // kColsBlock: the block's distances (null: the launch does not take this form)
  int last;         // and the level's last row
};

// The columns a launch reads on a level: the compact form when the context
// uses it and the level reads it (Level::read_compact), else the explicit
// indices.  block >= 0: the launch takes rows of that colour block alone.
//
// Where a block's slots have one distance each (has_block_offs), a launch reads the
// block's 27 distances, which stay in the caches, instead of a record for
// every slice.  V-cycles, records -> distances: 192^3 fp32 581 -> 548 us, 192^3
// kappa fp16 764 -> 709 (57 MB of records less), 64^3 245 -> 235.  Row runs keep the
// records (k_gs_run: 104^3 to 1e-9 32.0 ms with them, 33.5 without).
inline ColIdx col_idx(const Ctx *c, const Level &L, int block = -1) {
  ColIdx ci;
  ci.cols = L.cols;
  ci.cbase = ci.off = nullptr;
  if (!L.cbase || !((c->col_format == kColsCompact && L.read_compact) || c->col_format == kColsCompactAlways)) return ci;
  ci.cbase = L.cbase;
  ci.cdelta = L.cdelta;
  ci.cform = L.cform;
  if (block >= 0 && L.boffs) {
    ci.off = L.boffs + block * kMeta;
    ci.last = (int)(L.lay.npad - 1);
  }
  return ci;
}

// The value source and form of a launch.  The forms other than the stored
// array go with the compact columns: with explicit columns a launch reads the
// matrix as the reference stores it.
template <class VT, class ACC>
inline ValSrc<VT, ACC> val_src(const Level &L) {
  ValSrc<VT, ACC> v{nullptr, L.vmask, nullptr, L.field, L.diag_one ? 1 : 0};
  if constexpr (sizeof(VT) == 8) {
    v.vals = L.vals;
    v.slotv = L.slotv;
  } else if constexpr (sizeof(VT) == 4) {
    v.vals = L.vals32;
    if (L.slotv) v.slotv = reinterpret_cast<const float *>(L.slotv + kSlots);
  } else {
    v.vals = L.vals16;
    if (L.slotv) v.slotv = reinterpret_cast<const float *>(L.slotv + kSlots) + kSlots;
  }
  return v;
}
template <class VT>
inline int val_form(const Level &L, const ColIdx &ci) {
  if (!ci.cbase) return kValsStored;
  // the scaled fp16 values are one per slot only if the diagonals they are scaled by are
  if constexpr (sizeof(VT) == 2) return L.vform == kValsSlot && L.diag_one ? kValsSlot : kValsStored;
  else if constexpr (sizeof(VT) == 4) return L.vform == kValsSlot ? kValsSlot : kValsStored;
  else return L.vform;
}

// Runs f(CF, VF) with the column and value forms of a launch as constants.
// BLOCKS: the launch takes the rows of one block (col_idx was given it).
template <class VT, bool BLOCKS = false, class F>
inline void with_forms(const Level &L, const ColIdx &ci, F &&f) {
  if (!ci.cbase) return f(std::integral_constant<int, kColsStored>{}, std::integral_constant<int, kValsStored>{});
  const int vf = val_form<VT>(L, ci);
  auto with_vals = [&](auto CF) {
    if constexpr (sizeof(VT) == 8) {
      if (vf == kValsField) return f(CF, std::integral_constant<int, kValsField>{});
    }
    if (vf == kValsSlot) return f(CF, std::integral_constant<int, kValsSlot>{});
    f(CF, std::integral_constant<int, kValsStored>{});
  };
  if constexpr (BLOCKS) {
    if (ci.off) return with_vals(std::integral_constant<int, kColsBlock>{});
  }
  with_vals(std::integral_constant<int, kColsSlice>{});
}

// Slice of a row.  UNI: the 64 lanes of the wave hold the 64 rows of one
// slice (launches over 64-aligned rows), so the slice is wave-uniform and the
// per-slice metadata comes through the scalar cache.
template <bool UNI>
__device__ __forceinline__ int slice_of(int64_t row) {
  if constexpr (UNI) return __builtin_amdgcn_readfirstlane((int)(row >> 6));
  else return (int)(row >> 6);
}

// Column of (row, slot s).  CM 0: the explicit 32-bit index; CM 1: base +
// lane + int8 delta; CM 2: base + lane; CM 3: row + base (kColsBlock).  A launch picks one per slice
// (with_cols), so each inner loop is straight-line code; base holds the
// slice's 27 slot bases (with_cols provides them).
template <int CM, bool NT>
__device__ __forceinline__ int col_at(const ColIdx &ci, int64_t row, const int *base, size_t b, int s) {
  if constexpr (CM == 0) {
    return ld_col<NT>(ci.cols + b + s * kSlice);
  } else if constexpr (CM == 1) {
    int8_t d;
    if constexpr (NT) d = __builtin_nontemporal_load(ci.cdelta + b + s * kSlice);
    else d = ci.cdelta[b + s * kSlice];
    return base[s] + (int)(row & 63) + (int)d;
  } else if constexpr (CM == 2) {
    return base[s] + (int)(row & 63);
  } else {
    return min(max((int)row + base[s], 0), ci.last);  // the row of a slot without an entry may lie outside the level
  }
}

template <int V>
using cmode = std::integral_constant<int, V>;

// Runs f(cmode<CM>{}, base) with the column mode of the row's slice and its
// slot bases (kColsBlock: the distances).  UNI: the slice is the
// same for the whole wave: the bases and the form are read together from
// the slice's record before the choice, scalar loads in one round trip
// (small coarse steps are bound by their chain of dependent loads: reading
// the form first and the bases after it cost one more), and the choice is a
// scalar branch.  Otherwise each lane reads its slice's form from cform and
// its bases from the record as the slots need them.
template <int CF, bool UNI, class F>
__device__ __forceinline__ auto with_cols(const ColIdx &ci, int slice, F &&f) {
  if constexpr (CF == kColsStored) {
    return f(cmode<0>{}, (const int *)nullptr);
  } else if constexpr (CF == kColsBlock) {
    int off[kSlots];
#pragma unroll
    for (int s = 0; s < kSlots; ++s) off[s] = ci.off[s];
    return f(cmode<3>{}, (const int *)off);
  } else if constexpr (UNI) {
    const int *rec = ci.cbase + (int64_t)slice * kMeta;
    int base[kSlots];
#pragma unroll
    for (int s = 0; s < kSlots; ++s) base[s] = rec[s];
    const int form = rec[kSlots];
    if (form == kFormUniform) return f(cmode<2>{}, (const int *)base);
    if (form == kFormDelta) return f(cmode<1>{}, (const int *)base);
    return f(cmode<0>{}, (const int *)base);
  } else {
    const int *rec = ci.cbase + (int64_t)slice * kMeta;
    const int form = ci.cform[slice];
    if (form == kFormUniform) return f(cmode<2>{}, rec);
    if (form == kFormDelta) return f(cmode<1>{}, rec);
    return f(cmode<0>{}, rec);
  }
}

// A slot without an entry (a neighbour outside the grid) is a zero that names some
// other row, in the compact forms one far away in the grid: it adds an exact zero
// unless that row's x is NaN or infinite, or not written yet.  The row's sum is NaN
// then, and is taken again here over the entries alone, from the stored values and
// the explicit columns, which every level has.  start() is what the sum starts from
// (read again, so that no register holds it through the gathers).
//
// All other rows pay a compare and a branch that is not taken.  Solves, before ->
// after: 104^3 fp64 25.8 -> 25.8 ms, 192^3 fp64 42.3 -> 42.2, fp32 78.4 -> 76.5, kappa
// 256x192x144 fp16 111.2 -> 111.0, the adjoint at 128^3 (fp32, kappa) 96.5 -> 97.4.  A
// select in every product cost the first and the last two of these 1 to 3 %.
template <bool SUB, class VT, class XT, class ACC, class F>
__device__ __forceinline__ void mend_nan(ACC &sum, F &&start, const int *cols, const VT *vals, const XT *x, int64_t row,
                                         uint32_t mask) {
  if (__builtin_expect(__ballot(sum != sum) == 0, 1)) return;
  const bool again = sum != sum;
  if (again) sum = start();
#pragma unroll 1
  for (; mask; mask &= mask - 1) {
    const int s = __builtin_ctz(mask);
    const ACC a = ld_val<ACC, false>(vals + val_pos<val_width<VT>>(row, s));
    if (!again || a == (ACC)0) continue;
    const ACC t = a * (ACC)x[cols[ell_base(row) + s * kSlice]];
    if constexpr (SUB) sum -= t;
    else sum += t;
  }
}
// p[row] by a load of its own, whatever has been read from there before.
template <class T>
__device__ __forceinline__ T load_again(const T *p, int64_t row) {
  asm("" : "+v"(row));
  return p[row];
}
struct FromZero {
  __device__ int operator()() const { return 0; }
};

// ---------------------------------------------------------------------------
// deterministic reductions: fixed partition, fixed tree, last block finishes

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
  return v;
}

// Deterministic reductions in two kernels.  Each block of the producing
// kernel reduces its values in a fixed tree (shuffles, then 4 waves in order)
// and stores one partial per value with a plain store; a one-block finishing
// kernel then sums the partials in a fixed order and applies the scalar
// update.  Within a kernel no fences or atomics are needed: the kernel
// boundary makes the partials visible (an agent-scope fence inside a kernel
// writes back or invalidates the whole L2 of an XCD, which costs far more
// than the extra launch).
template <int NV>
__device__ __forceinline__ void block_partials(const double (&v)[NV], double *partials) {
  __shared__ double sh[4][NV];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    const double s = wave_sum(v[k]);
    if (lane == 0) sh[w][k] = s;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
#pragma unroll
    for (int k = 0; k < NV; ++k)
      partials[(size_t)k * gridDim.x + blockIdx.x] = (sh[0][k] + sh[1][k]) + (sh[2][k] + sh[3][k]);
  }
}

// What the finishing kernel does with the totals (t0, t1).  F_DOT and F_NORMR2
// also leave t0 in pinned host memory where the host waits for it (host,
// wait_host); a copy behind the kernel and a wait for the stream took 6 us more
// per answer (dot, WAXPBY, WAXPBY + dot at 48^3: 56 -> 43 us).
enum FinishOp : int {
  F_DOT = 0,        // scal[S_DOT] = t0
  F_RZ_FIRST,       // rtz = t0                                   (CG.cpp:110)
  F_RZ,             // oldrtz = rtz; rtz = t0; beta = rtz/oldrtz  (CG.cpp:112-114)
  F_PAP,            // pAp = t0; alpha = rtz/pAp                  (CG.cpp:119-120)
  F_NORMR2,         // normr^2 = t0                               (CG.cpp:123)
                    // with a slot: record t0 there; stop test t0 > 0
  F_FCG,            // oldrtz = rtz; rtz = t0; beta = -alpha t1 / oldrtz
};

// The store must reach the host while it polls, so it has system scope.  It
// orders nothing else: whatever the total stands for was written by kernels
// before this one.
__device__ __forceinline__ void give_host(double *host, double v) {
  __hip_atomic_store(host, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

constexpr int kFinishThreads = 1024;
constexpr int kFinishLoads = 32;  // partials per finishing thread read in one round

// Reductions over more than kFoldAbove partials first fold each run of kFold
// consecutive partials into one (one block per run), so the one-block
// finishing kernel reads few values: its single CU would otherwise take
// ~100 us over the 524288 partials of a 512^3 pass.
constexpr int64_t kFold = 4096;
constexpr int64_t kFoldAbove = 32768;

template <int NV>
__global__ __launch_bounds__(kBlock) void k_fold(const double *__restrict__ in, int64_t G, double *out) {
  double v[NV];
  const int64_t b0 = (int64_t)blockIdx.x * kFold;
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    const double *p = in + (size_t)k * G;
    double a0 = 0.0, a1 = 0.0;
#pragma unroll 4
    for (int64_t j = threadIdx.x; j < kFold; j += 2 * kBlock) {
      const int64_t i = b0 + j;
      if (i < G) a0 += p[i];
      if (i + kBlock < G) a1 += p[i + kBlock];
    }
    v[k] = a0 + a1;
  }
  block_partials<NV>(v, out);
}

template <int NV>
__global__ __launch_bounds__(kFinishThreads) void k_finish(const double *__restrict__ partials, int64_t G,
                                                           double *scal, int op, double *slot, double *host) {
  __shared__ double sh[kFinishThreads / 64][NV];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    const double *p = partials + (size_t)k * G;
    double a0 = 0.0, a1 = 0.0, a2 = 0.0, a3 = 0.0;
    constexpr int64_t T = kFinishThreads;
    const int64_t tid = threadIdx.x;
    if (G <= kFinishLoads * T) {
      // The additions of the loop below, in the same order into the same
      // accumulators, with all loads issued first: one round trip to memory
      // instead of one per group of four.  Element j of this thread is
      // p[tid + j T]; the loop adds it to a(j % 4) in group j / 4 while the
      // group's last element is below G, then the rest to a0.
      double v[kFinishLoads];
#pragma unroll
      for (int j = 0; j < kFinishLoads; ++j) {
        const int64_t i = tid + j * T;
        v[j] = i < G ? p[i] : 0.0;
      }
      const int64_t ngroups = G > tid + 3 * T ? (G - tid - 3 * T - 1) / (4 * T) + 1 : 0;
      const int64_t nmine = G > tid ? (G - tid - 1) / T + 1 : 0;
#pragma unroll
      for (int j = 0; j < kFinishLoads; ++j) {
        if (j / 4 < ngroups) {
          if (j % 4 == 0) a0 += v[j];
          else if (j % 4 == 1) a1 += v[j];
          else if (j % 4 == 2) a2 += v[j];
          else a3 += v[j];
        } else if (j < nmine) {
          a0 += v[j];
        }
      }
    } else {
      int64_t i = tid;
      for (; i + 3 * T < G; i += 4 * T) {
        a0 += p[i];
        a1 += p[i + T];
        a2 += p[i + 2 * T];
        a3 += p[i + 3 * T];
      }
      for (; i < G; i += T) a0 += p[i];
    }
    const double s = wave_sum((a0 + a1) + (a2 + a3));
    if (lane == 0) sh[w][k] = s;
  }
  __syncthreads();
  if (threadIdx.x != 0) return;
  double t[NV];
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    double s = 0.0;
    for (int j = 0; j < kFinishThreads / 64; ++j) s += sh[j][k];
    t[k] = s;
  }
  switch (op) {
    case F_DOT:
      scal[S_DOT] = t[0];
      if (host) give_host(host, t[0]);
      break;
    case F_RZ_FIRST: scal[S_RTZ] = t[0]; break;
    case F_RZ: {
      const double old = scal[S_RTZ];
      scal[S_OLDRTZ] = old;
      scal[S_RTZ] = t[0];
      scal[S_BETA] = t[0] / old;
      break;
    }
    case F_PAP:
      scal[S_PAP] = t[0];
      scal[S_ALPHA] = scal[S_RTZ] / t[0];
      break;
    case F_NORMR2:
      // Deferred stop test of a tolerance-0 solve (CG.cpp:100 with tolerance
      // 0): with normr0 finite and positive, normr/normr0 > 0 holds exactly
      // when normr^2 > 0.  The first norm that fails (zero or NaN) raises
      // S_STOP; from then on k_cg_update leaves x and r alone and no norm
      // is recorded.  Without a slot the flag is cleared (solver preamble).
      if (slot) {
        if (scal[S_STOP] != 0.0) break;
        *slot = t[0];
        if (!(t[0] > 0.0)) scal[S_STOP] = 1.0;
      } else {
        scal[S_STOP] = 0.0;
      }
      scal[S_NORMR2] = t[0];
      if (host) give_host(host, t[0]);
      break;
    case F_FCG: {
      const double old = scal[S_RTZ];
      scal[S_OLDRTZ] = old;
      scal[S_RTZ] = t[0];
      scal[S_BETA] = -scal[S_ALPHA] * t[NV - 1] / old;
      break;
    }
  }
}

// Streaming reductions give each block one chunk of kChunk * kBlock
// consecutive elements, kChunk per thread, each a coalesced wave access.
constexpr int kChunk = 4;
__device__ __forceinline__ int64_t chunk_index(int j) {
  return ((int64_t)blockIdx.x * kChunk + j) * kBlock + threadIdx.x;
}

// ---------------------------------------------------------------------------
// sparse kernels (one thread per row, 4 slices per block)

// ---------------------------------------------------------------------------
// Row runs: two consecutive fp64 rows per lane (kValsSlot and kValsField)
//
// Without the value stream a large pass is bound by the vector L1: it takes
// a load of 64 lanes in 16 steps of four lanes whether a lane asks for 8 or 16
// bytes (measured: 17 L1 accesses per 8-byte gather; on a 512^3 fine step the
// address units were busy for 80 % of the time).  So a lane takes two
// consecutive rows and gathers each slot's two neighbours with one 16-byte
// load: in a uniform slice they are consecutive.  The wave covers two slices;
// it takes this path where the second continues the first (k_slice_runs: both
// uniform, each slot's base going on by 64), which holds but for a few slices
// at the ends of blocks and strips; elsewhere it takes its slices one after
// the other, a row per lane.  Products and sums of a row are the same, in the
// same order.
//
// kValsSlot, a row per lane -> runs: 512^3 fine step 369 -> 301 us (1.6 GB,
// 5.3 TB/s), 192^3 17.9 -> 14.7 us, 192^3 SpMV 113 -> 77 us; kValsField: 128^3
// fine step 10.7 -> 9.0 us.  The fp32 and fp16 passes keep a row per lane:
// 192^3 fine step 10.6 us, 11.0 with two rows and 11.6 with four.
//
// Launches of fewer rows keep it too (a wave of a run needs longer, with twice
// the sums, and a small launch waits for its last wave): without / with runs,
// 104^3 fine steps (140608 rows) 5.9 / 5.8 us, 96^3 (110592) 4.6 / 4.4, 48^3
// (13824) 3.2 / 4.0.
constexpr int64_t kRunMinRows = 1 << 17;

// Whether a launch over `rows` rows of a level takes row runs.
inline bool run_rows(const Level &L, int64_t rows) { return L.runs && rows >= kRunMinRows; }

typedef double f64x2_u __attribute__((ext_vector_type(2), aligned(8)));
__device__ __forceinline__ void ld_pair(const double *p, double (&v)[2]) {
  const f64x2_u t = *reinterpret_cast<const f64x2_u *>(p);
  v[0] = t.x;
  v[1] = t.y;
}
__device__ __forceinline__ void st_pair(double *p, const double (&v)[2]) {
  f64x2_u t;
  t.x = v[0];
  t.y = v[1];
  *reinterpret_cast<f64x2_u *>(p) = t;
}

// Whether the next slice continues a slice, in the slice's record.
constexpr int kRunAt = kSlots + 1;

// The off-diagonal values' inputs and the diagonals of a lane's two rows.
template <int VF>
struct RunVals {
  uint32_t m[2];
  double d[2], ki[2];
  __device__ __forceinline__ void load(const ValSrc<double, double> &src, int64_t row) {
    const u32x2_t t = *reinterpret_cast<const u32x2_t *>(src.mask + row);
    m[0] = t.x;
    m[1] = t.y;
    if (VF == kValsSlot && src.diag_one) {
#pragma unroll
      for (int j = 0; j < 2; ++j) d[j] = (m[j] >> kDiagSlot) & 1u ? src.slotv[kDiagSlot] : 1.0;
    } else {  // the diagonals of a slice are adjacent
      ld_pair(src.vals + val_pos<2>(row, kDiagSlot), d);
    }
    if constexpr (VF == kValsField) ld_pair(src.field + row, ki);
  }
};

// sum[j] += (SUB: -=) a x over the slots in MASK, ascending.  base: the
// first slice's slot bases (scalars); e0: the lane's first row, from the
// run's start; row: the lane's first row; xd: x of the rows themselves; r: what the
// sums start from, if not 0.
template <int VF, uint32_t MASK, bool SUB>
__device__ __forceinline__ void run_sum(const int *cols, const int (&base)[kSlots], unsigned e0,
                                        const ValSrc<double, double> &src, const RunVals<VF> &v,
                                        const double *r, const double *__restrict__ x, int64_t row,
                                        const double (&xd)[2], double (&sum)[2]) {
#pragma unroll
  for (int s = 0; s < kSlots; ++s) {
    if (!((MASK >> s) & 1u)) continue;
    double xv[2] = {xd[0], xd[1]}, kv[2];
    if (s != kDiagSlot) {
      ld_pair(x + base[s] + e0, xv);
      if constexpr (VF == kValsField) ld_pair(src.field + base[s] + e0, kv);
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      double a;
      if (s == kDiagSlot) a = v.d[j];
      else if constexpr (VF == kValsField) a = bit_select(v.m[j], s, -((v.ki[j] + kv[j]) * 0.5));
      else a = bit_select(v.m[j], s, src.slotv[s]);
      const double t = a * xv[j];
      if constexpr (SUB) sum[j] -= t;
      else sum[j] += t;
    }
  }
#pragma unroll
  for (int j = 0; j < 2; ++j)
    mend_nan<SUB>(sum[j], [&] { return SUB ? load_again(r, row + j) : 0.0; }, cols, src.vals, x, row + j, MASK);
}

// A wave's place in a launch over the 64-row slices of [row0, row0 + nrows),
// nrows a multiple of 64: it takes the slices 2g and 2g + 1 of it.  On a run
// the lane's rows are row + 2 lane and the next one (active: it has rows),
// else row + 64 j + lane of slice j.
struct RunWave {
  int64_t row;  // first row of the wave
  int slices;   // slices it takes (0: past the end)
  bool run, active;
  int base[kSlots];
  __device__ __forceinline__ void init(const ColIdx &ci, int64_t row0, int64_t nrows, int64_t tile) {
    const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    take(ci, row0, nrows, (tile * (int64_t)(blockDim.x >> 6) + w) * 2);
  }
  // slices g and g + 1 of the launch
  __device__ __forceinline__ void take(const ColIdx &ci, int64_t row0, int64_t nrows, int64_t g) {
    const int64_t left = (nrows >> 6) - g;
    row = row0 + g * kSlice;
    slices = left <= 0 ? 0 : left < 2 ? 1 : 2;
    run = active = false;
    if (slices) {
      const int *rec = ci.cbase + (row >> 6) * kMeta;
#pragma unroll
      for (int s = 0; s < kSlots; ++s) base[s] = rec[s];
      run = rec[kSlots] == kFormUniform && rec[kRunAt] >= slices - 1;
      active = run && 2 * (threadIdx.x & 63) < (unsigned)slices * kSlice;
    }
  }
  __device__ __forceinline__ int64_t lane_row(int j) const {
    const unsigned lane = threadIdx.x & 63;
    return run ? row + 2 * lane + j : row + j * kSlice + lane;
  }
  __device__ __forceinline__ bool has_row(int j) const { return run ? active : j < slices; }
};

// a[j] = v for a j known at run time, the array kept in registers.
__device__ __forceinline__ void put(double (&a)[2], int j, double v) {
  a[0] = j == 0 ? v : a[0];
  a[1] = j == 1 ? v : a[1];
}

// Workgroups of a row-run launch per colour block, where level_tile can take the
// blocks together: equal ones, a multiple of 8 workgroups each (else 0).
inline int block_tiles(const Level &L) {
  const int64_t rows = L.lay.start[1];
  for (int k = 0; k < kColours; ++k)
    if (L.lay.start[k + 1] - L.lay.start[k] != rows) return 0;
  return rows % (8 * 2 * kBlock) ? 0 : (int)(rows / (2 * kBlock));
}
// Workgroups of a row-run launch over `rows` rows.
inline unsigned run_tiles(int64_t rows, int bs = kBlock) { return (unsigned)((rows + 2 * bs - 1) / (2 * bs)); }

// y = A x over rows [0, nrows); ComputeSPMV_ref.cpp:61-70
template <class VT, class XT, class ACC, int CF, int VF>
__global__ __launch_bounds__(kBlock) HPCGX_SPARSE_OCCUPANCY(VT, CF) void k_spmv(const ColIdx ci,
                                                 const ValSrc<VT, ACC> src,
                                                 const XT *__restrict__ x, XT *__restrict__ y,
                                                 int64_t nrows) {
  const int64_t row = tile_id() * kBlock + threadIdx.x;
  if (row >= nrows) return;
  const size_t b = ell_base(row);
  const int slice = slice_of<true>(row);
  RowVals<VF, VT, ACC, true, kAllSlots> v;
  v.load(src, row);
  ACC ax = with_cols<CF, true>(ci, slice, [&](auto cm, const int *base) {
    constexpr int CM = decltype(cm)::value;
    ACC sum = 0;
#pragma unroll
    for (int s = 0; s < kSlots; ++s) {
      const int c = col_at<CM, true>(ci, row, base, b, s);
      sum += v.at(s, c) * (ACC)x[c];
    }
    return sum;
  });
  mend_nan<false>(ax, FromZero{}, ci.cols, src.vals, x, row, kAllSlots);
  y[row] = (XT)ax;
}

// (A x) of a wave's rows (RunWave::lane_row), 0 where a lane has none.
template <int VF>
__device__ __forceinline__ void run_ax(const ColIdx &ci, const ValSrc<double, double> &src, const RunWave &w,
                                       const double *__restrict__ x, double (&out)[2]) {
  const unsigned lane = threadIdx.x & 63;
  out[0] = out[1] = 0.0;
  if (w.run) {
    if (!w.active) return;
    RunVals<VF> v;
    v.load(src, w.row + 2 * lane);
    double xd[2];
    ld_pair(x + w.row + 2 * lane, xd);
    run_sum<VF, kAllSlots, false>(ci.cols, w.base, 2 * lane, src, v, nullptr, x, w.row + 2 * lane, xd, out);
    return;
  }
#pragma unroll 1
  for (int j = 0; j < w.slices; ++j) {
    const int64_t row = w.row + j * kSlice + lane;
    RowVals<VF, double, double, false, kAllSlots> v;
    v.load(src, row);
    double ax = with_cols<kColsSlice, true>(ci, slice_of<true>(row), [&](auto cm, const int *base) {
      constexpr int CM = decltype(cm)::value;
      double sum = 0;
#pragma unroll
      for (int s = 0; s < kSlots; ++s) {
        const int c = col_at<CM, true>(ci, row, base, ell_base(row), s);
        sum += v.at(s, c) * x[c];
      }
      return sum;
    });
    mend_nan<false>(ax, FromZero{}, ci.cols, src.vals, x, row, kAllSlots);
    put(out, j, ax);
  }
}

// y = A x by row runs
template <int VF>
__global__ __launch_bounds__(kBlock) void k_spmv_run(const ColIdx ci, const ValSrc<double, double> src,
                                                     const double *__restrict__ x, double *__restrict__ y,
                                                     int64_t nrows, int bt) {
  RunWave w;
  w.init(ci, 0, nrows, level_tile(bt));
  if (!w.slices) return;
  double ax[2];
  run_ax<VF>(ci, src, w, x, ax);
  if (w.run) {
    if (w.active) st_pair(y + w.lane_row(0), ax);
  } else {
#pragma unroll
    for (int j = 0; j < 2; ++j)
      if (w.has_row(j)) y[w.lane_row(j)] = ax[j];
  }
}

// Slots whose neighbour lies in a block swept before block k in the default
// order (the neighbour at offset d has class c ^ oddness(d)).
__host__ __device__ constexpr uint32_t swept_before_mask(int k) {
  int pos[kColours] = {};
  for (int j = 0; j < kColours; ++j) pos[kDefaultOrder[j]] = j;
  uint32_t m = 0;
  for (int s = 0; s < kSlots; ++s) {
    const int odd = ((s % 3) != 1) | ((((s / 3) % 3) != 1) << 1) | (((s / 9) != 1) << 2);
    if (pos[kDefaultOrder[k] ^ odd] < k) m |= 1u << s;
  }
  return m;
}

// The masks keep or skip the slots of a unit together (each unit's
// neighbours lie in one colour block).
constexpr bool masks_keep_units(int W) {
  for (int k = 0; k < kColours; ++k)
    for (int u = 0; u < val_units(W); ++u) {
      const uint32_t um = unit_mask(val_unit(W, u)), m = swept_before_mask(k) & um;
      if (m != 0 && m != um) return false;
    }
  return true;
}
static_assert(masks_keep_units(2) && masks_keep_units(4), "zero-start masks split a value unit");

#ifndef HPCGX_FINE_ROT
#define HPCGX_FINE_ROT 1
#endif

// One Gauss-Seidel step on the rows of one colour block; ComputeSYMGS_ref.cpp:72-79:
// sum = r_i - sum_j a_ij x_j (diagonal included) + x_i a_ii ; x_i = sum / a_ii.
// ZK >= 0: the step of block ZK in the first forward sweep from x = 0 -- only
// neighbours in blocks swept before ZK can be nonzero; the other terms are
// exact zeros and are not read, and neither is x_i (x may hold anything on
// entry).  The skipped set is a compile-time constant, so the remaining loads
// issue back to back.
// FINE: the finest level (streamed matrix loads; its own instantiation, so
// profiles show the dominant launches separately from the coarse levels').
// ZK == 0 reads no neighbour at all (x_i = r_i / a_ii), which holds for the
// first block of any order, general levels included.
// GEN: general level, the diagonal's slot is dslot[row] (stencil: slot 13).
// gs_value is a row's new value; gs_row the update of one row, which
// returns r_i * x_i (new) for the fused r.z.
template <class VT, class XT, class ACC, int ZK, bool FINE, int CF, int VF, bool GEN>
__device__ __forceinline__ XT gs_value(const ColIdx &ci, const ValSrc<VT, ACC> &src, const XT *r, const XT *x,
                                       int64_t row, const uint8_t *__restrict__ dslot) {
  constexpr uint32_t mask = ZK >= 0 ? swept_before_mask(ZK) : kAllSlots;
  const size_t b = ell_base(row);
  const int slice = slice_of<true>(row);
  RowVals<VF, VT, ACC, FINE, mask> vr;
  vr.load(src, row);
  ACC d;
  if constexpr (!GEN) d = vr.diag(src, row);
  else d = ld_val<ACC, FINE>(src.vals + val_pos<val_width<VT>>(row, (int)dslot[row]));
  const ACC xi = ZK < 0 ? (ACC)x[row] : (ACC)0;
  auto row_sum = [&](auto cm, const int *base) {
    constexpr int CM = decltype(cm)::value;
    ACC sum = (ACC)r[row];
#pragma unroll
    for (int s = 0; s < kSlots; ++s) {
      if (!((mask >> s) & 1u)) continue;
      if (!GEN && CF != kColsStored && s == kDiagSlot) {  // explicit columns: every index is read, its own too
        sum -= vr.at(s, 0) * xi;
        continue;
      }
      const int c = col_at<CM, FINE>(ci, row, base, b, s);
      sum -= vr.at(s, c) * (ACC)x[c];
    }
    return sum;
  };
  ACC sum = with_cols<CF, true>(ci, slice, row_sum);
  // not on general levels: their slots without an entry name the row itself or its
  // slice's neighbourhood
  if constexpr (!GEN) mend_nan<true>(sum, [&] { return load_again(r, row); }, ci.cols, src.vals, x, row, mask);
  if (ZK < 0) sum += xi * d;
  return (XT)(sum / d);
}

template <class VT, class XT, class ACC, int ZK, bool FINE, int CF, int VF, bool GEN>
__device__ __forceinline__ double gs_row(const ColIdx &ci, const ValSrc<VT, ACC> &src,
                                         const XT *__restrict__ r, XT *__restrict__ x, int64_t row,
                                         const uint8_t *__restrict__ dslot) {
  const XT xn = gs_value<VT, XT, ACC, ZK, FINE, CF, VF, GEN>(ci, src, r, x, row, dslot);
  x[row] = xn;
  return (double)r[row] * (double)xn;
}

// RZ: this step writes the final value of its rows in the V-cycle (the
// post-smoother's last forward block and its backward steps); the block
// also leaves its partial sum of r_i x_i in rz[blockIdx.x], so the solver's
// r.z needs no pass of its own.
template <class VT, class XT, class ACC, int ZK, bool FINE, int CF = kColsStored, int VF = kValsStored, bool GEN = false,
          bool RZ = false>
__global__ __launch_bounds__(kBlock)
__attribute__((amdgpu_waves_per_eu(1, SparseOccupancy<VT, CF, ZK < 0 ? kSlots : __builtin_popcount(swept_before_mask(ZK))>::max_waves)))
void k_gs(const ColIdx ci, const ValSrc<VT, ACC> src,
                                               const XT *__restrict__ r, XT *__restrict__ x,
                                               int64_t row0, int64_t nrows,
                                               const uint8_t *__restrict__ dslot, double *rz = nullptr) {
  static_assert(!GEN || ZK <= 0, "general levels: full rows, or the first block from x = 0 (diagonal only)");
  static_assert(!RZ || ZK < 0, "r.z is taken from the post-smoother");
  static_assert(VF == kValsStored || (CF && !GEN), "value forms: stencil levels with compact columns");
  // blocks of 256 threads, or of 64 for small steps (one wave per block
  // spreads them over more CUs: gs_block); the r.z form always takes 256
  const int64_t t = tile_id<HPCGX_FINE_ROT && FINE && sizeof(VT) == 8>() * (int64_t)blockDim.x + threadIdx.x;
  if constexpr (RZ) {
    // every thread reaches the block reduction; rows past the block add 0
    double acc = 0.0;
    if (t < nrows) acc = gs_row<VT, XT, ACC, ZK, FINE, CF, VF, GEN>(ci, src, r, x, row0 + t, dslot);
    const double v[1] = {acc};
    block_partials<1>(v, rz);
    return;
  }
  if (t >= nrows) return;
  gs_row<VT, XT, ACC, ZK, FINE, CF, VF, GEN>(ci, src, r, x, row0 + t, dslot);
}

// The partial sums of a value per row, as the one-row-per-lane launch leaves
// them: v[j] belongs to row lane_row(j).  Each 64-row slice is reduced over row
// distances 32, 16, .. 1 as wave_sum does it, and the four slices of a 256-row
// tile as block_partials does; the tile's sum goes where that launch's block
// would leave it.  ntiles: tiles of the launch.
template <bool ROT>
__device__ __forceinline__ void run_partials(const RunWave &w, double (&v)[2], int64_t tile, int64_t ntiles,
                                             double *partials) {
  __shared__ double sh[2 * kBlock / kSlice];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (w.run) {  // lanes 0..31 hold the first slice's rows, two each
#pragma unroll
    for (int off = 16; off > 0; off >>= 1) {
      v[0] += __shfl_down(v[0], off, 64);
      v[1] += __shfl_down(v[1], off, 64);
    }
    if ((lane & 31) == 0) sh[2 * wave + (lane >> 5)] = v[0] + v[1];
  } else {
    const double a = wave_sum(v[0]), b = wave_sum(v[1]);
    if (lane == 0) {
      sh[2 * wave] = a;
      sh[2 * wave + 1] = b;
    }
  }
  __syncthreads();
  if (threadIdx.x < 2) {
    const int64_t t = 2 * tile + threadIdx.x;
    const double *q = sh + 4 * threadIdx.x;
    if (t < ntiles) partials[tile_slot<ROT>((unsigned)t, (unsigned)ntiles)] = (q[0] + q[1]) + (q[2] + q[3]);
  }
}

// One Gauss-Seidel step on a wave's two slices; acc[j]: r_i x_i of lane_row(j).
template <int ZK, bool FINE, int VF>
__device__ __forceinline__ void gs_run_rows(const ColIdx &ci, const ValSrc<double, double> &src, const RunWave &w,
                                            const double *__restrict__ r, double *x, double (&acc)[2]) {
  constexpr uint32_t mask = ZK >= 0 ? swept_before_mask(ZK) : kAllSlots;
  acc[0] = acc[1] = 0.0;
  if (w.run) {
    if (!w.active) return;
    const int64_t row = w.lane_row(0);
    RunVals<VF> v;
    v.load(src, row);
    double rv[2], xd[2] = {0.0, 0.0}, xn[2];
    ld_pair(r + row, rv);
    if constexpr (ZK < 0) ld_pair(x + row, xd);
    double sum[2] = {rv[0], rv[1]};
    run_sum<VF, mask, true>(ci.cols, w.base, 2 * (threadIdx.x & 63), src, v, r, x, row, xd, sum);
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      if constexpr (ZK < 0) sum[j] += xd[j] * v.d[j];
      xn[j] = sum[j] / v.d[j];
      acc[j] = rv[j] * xn[j];
    }
    st_pair(x + row, xn);
    return;
  }
#pragma unroll 1
  for (int j = 0; j < w.slices; ++j)
    put(acc, j, gs_row<double, double, double, ZK, FINE, kColsSlice, VF, false>(ci, src, r, x, w.lane_row(j), nullptr));
}

// One Gauss-Seidel step by row runs (k_gs on kValsSlot and kValsField levels).
template <int ZK, bool FINE, int VF, bool RZ = false>
__global__ __launch_bounds__(kBlock) void k_gs_run(const ColIdx ci, const ValSrc<double, double> src,
                                                   const double *__restrict__ r, double *__restrict__ x,
                                                   int64_t row0, int64_t nrows, double *rz = nullptr) {
  constexpr bool ROT = HPCGX_FINE_ROT && FINE;
  const int64_t tile = tile_id<ROT>();
  RunWave w;
  w.init(ci, row0, nrows, tile);
  double acc[2];
  gs_run_rows<ZK, FINE, VF>(ci, src, w, r, x, acc);
  if constexpr (RZ) run_partials<ROT>(w, acc, tile, (nrows + kBlock - 1) / kBlock, rz);
}

// Colour steps that follow one another on two classes that differ in x alone (4
// then 5, and 1, 0, 1 around the turn of the sweep), in one launch.
//
// Rows of the two classes couple only along their own grid line: a launch in
// which each workgroup takes whole lines of both blocks, with a barrier in
// place of the launch between the steps, updates every row from the values that
// the separate steps would read.  A launch less is 3 to 4 us less where a step
// is bound by its own latency; see lines_pay for where that ends.  V-cycles,
// steps apart -> these pairs -> and those in z (k_gs_columns): 64^3 fp64 234 -> 208 ->
// 199 us, 104^3 371 -> 326 -> 324, 128^3 fp32 376 -> 325 -> 302, kappa 104^3 fp16 342 ->
// 299 -> 293.
//
// Past the end of a line, the slots along it name another line of the other
// block, which another workgroup may be updating: times the slot's zero that adds
// nothing, whichever value is read (mend_nan, should it be NaN).
//
// A row per lane, columns by the blocks' distances; a workgroup takes `rows`
// rows (whole lines) of each block.  STEPS 3: the first block again.  ZA, ZB: the
// steps' places in a sweep from x = 0 (ZK of k_gs), or -1.
template <class VT, class XT, class ACC, int ZA, int ZB, int STEPS, bool FINE, int VF>
__global__ __launch_bounds__(kBlock) void k_gs_lines(const ColIdx cia, const ColIdx cib, const ValSrc<VT, ACC> src,
                                                     const XT *__restrict__ r, XT *x, int64_t rowa, int64_t rowb,
                                                     int64_t nrows, int rows) {
  const int64_t i = tile_id() * rows + threadIdx.x;
  const bool in = (int)threadIdx.x < rows && i < nrows;
  auto step = [&](auto zk, const ColIdx &ci, int64_t row) {
    if (in)
      x[row] = gs_value<VT, XT, ACC, decltype(zk)::value, FINE, kColsBlock, VF, false>(ci, src, r, x, row, nullptr);
  };
  step(std::integral_constant<int, ZA>{}, cia, rowa + i);
  __syncthreads();
  step(std::integral_constant<int, ZB>{}, cib, rowb + i);
  if constexpr (STEPS == 3) {
    __syncthreads();
    step(std::integral_constant<int, -1>{}, cia, rowa + i);
  }
}

// The same for two classes that differ in z alone (7 then 3, 2 then 6, and
// back): their rows couple only along z, and a workgroup takes `cols` columns of
// both blocks through all nz planes of `plane` rows; one more takes the rows that
// pad the blocks.  Workgroups of 512 threads were slower (64^3 223 us).
template <class VT, class XT, class ACC, int ZA, int ZB, bool FINE, int VF>
__global__ __launch_bounds__(kBlock) void k_gs_columns(const ColIdx cia, const ColIdx cib, const ValSrc<VT, ACC> src,
                                                       const XT *__restrict__ r, XT *x, int64_t rowa, int64_t rowb,
                                                       int64_t nrows, int plane, int nz, int cols) {
  const int64_t tile = tile_id();
  const int z = (int)threadIdx.x / cols;
  const int64_t q = tile * cols + ((int)threadIdx.x - z * cols);
  bool in = z < nz && q < plane;
  int64_t i = (int64_t)z * plane + q;
  if (tile * cols >= plane) {
    i = (int64_t)nz * plane + threadIdx.x;
    in = i < nrows;
  }
  auto step = [&](auto zk, const ColIdx &ci, int64_t row) {
    if (in)
      x[row] = gs_value<VT, XT, ACC, decltype(zk)::value, FINE, kColsBlock, VF, false>(ci, src, r, x, row, nullptr);
  };
  step(std::integral_constant<int, ZA>{}, cia, rowa + i);
  __syncthreads();
  step(std::integral_constant<int, ZB>{}, cib, rowb + i);
}

// Residual at the injected rows and restriction, fused (ComputeMG_ref.cpp:49-51 +
// ComputeRestriction_ref.cpp:51): rc[inj[t]] = r_f - (A x)_f for the t-th
// injected row f = row0 + t (frow[t] when frow is given).  (A x)_f is summed
// from 0 like SpMV, then subtracted.  SCALE: fp16 V-cycle, times sigma[t].
template <class VT, class XT, class ACC, bool SCALE, int CF, int VF>
__global__ __launch_bounds__(kBlock) HPCGX_SPARSE_OCCUPANCY(VT, CF) void k_restrict(const ColIdx ci, const ValSrc<VT, ACC> src,
                                                     const XT *__restrict__ r,
                                                     const XT *__restrict__ x,
                                                     XT *__restrict__ rc, const int *__restrict__ inj,
                                                     const float *__restrict__ sigma, int64_t row0,
                                                     int64_t count, const int *__restrict__ frow) {
  const int64_t t = tile_id() * kBlock + threadIdx.x;
  if (t >= count) return;
  const int64_t row = frow ? (int64_t)frow[t] : row0 + t;
  const size_t b = ell_base(row);
  RowVals<VF, VT, ACC, true, kAllSlots> v;
  v.load(src, row);
  auto row_ax = [&](auto cm, const int *base) {
    constexpr int CM = decltype(cm)::value;
    ACC ax = 0;
#pragma unroll
    for (int s = 0; s < kSlots; ++s) {
      const int c = col_at<CM, true>(ci, row, base, b, s);
      ax += v.at(s, c) * (ACC)x[c];
    }
    return ax;
  };
  ACC ax;
  if (frow) {  // rows from a list: slices differ across the wave
    const int slice = slice_of<false>(row);
    ax = with_cols<CF, false>(ci, slice, row_ax);
  } else {
    const int slice = slice_of<true>(row);
    ax = with_cols<CF, true>(ci, slice, row_ax);
  }
  mend_nan<false>(ax, FromZero{}, ci.cols, src.vals, x, row, kAllSlots);
  ACC res = (ACC)r[row] - ax;
  if (SCALE) res = res * (ACC)sigma[t];
  rc[inj[t]] = (XT)res;
}

// k_restrict over the block of injected rows by row runs; the rows that pad
// the block to whole slices are not written.
template <int VF>
__global__ __launch_bounds__(kBlock) void k_restrict_run(const ColIdx ci, const ValSrc<double, double> src,
                                                         const double *__restrict__ r, const double *__restrict__ x,
                                                         double *__restrict__ rc, const int *__restrict__ inj,
                                                         int64_t row0, int64_t count) {
  RunWave w;
  w.init(ci, row0, (count + kSlice - 1) / kSlice * kSlice, tile_id());
  if (!w.slices) return;
  double ax[2];
  run_ax<VF>(ci, src, w, x, ax);
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int64_t row = w.lane_row(j), t = row - row0;
    if (w.has_row(j) && t < count) rc[inj[t]] = r[row] - ax[j];
  }
}

// x_f += xc at the injected rows (ComputeProlongation_ref.cpp:49).
template <class XT, class ACC, bool SCALE>
__global__ __launch_bounds__(kBlock) void k_prolong(XT *__restrict__ x, const XT *__restrict__ xc,
                                                    const int *__restrict__ inj,
                                                    const float *__restrict__ sigma, int64_t row0,
                                                    int64_t count, const int *__restrict__ frow) {
  const int64_t t = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (t >= count) return;
  const int64_t row = frow ? (int64_t)frow[t] : row0 + t;
  ACC v = (ACC)xc[inj[t]];
  if (SCALE) v = v * (ACC)sigma[t];
  x[row] = (XT)((ACC)x[row] + v);
}

// ---------------------------------------------------------------------------
// The tail of the V-cycle in one workgroup
//
// A colour step of a small level takes a launch 2 to 4 us whatever its size
// (start-up, a chain of dependent loads and sums, draining), and a V-cycle has
// 15 or 30 of them per level.  From the first level of up to kTailRows rows
// on, one workgroup runs the rest of the V-cycle: x and r live in LDS, a
// barrier separates the colour steps, the matrix comes from L2.  The rows' sums
// are those of the separate launches, in the same order.
//
// V-cycles, called back to back, launches -> tail -> with sweep_slot: 8^3 (3 levels)
// 151 -> 81 -> 70 us, 16^3 (4 levels) 220 -> 124 -> 105 (fp32 225 -> 133 -> 94), 20^3 (2
// levels) 94 -> 82 -> 73 (fp32 100 -> 79 -> 64).  The limit is a block of
// a slice per wave: a 24^3 level (27 slices a block) takes one CU as long as a
// launch per step takes 256 (64 us against 47 to 57), a 26^3 one longer (187
// against 132).
constexpr int kTailRows = 8192;       // padded rows of the tail's first level
constexpr int kTailThreads = 1024;
constexpr int kTailColours = 16;      // colours of a level it can sweep
constexpr int kTailLds = 160 * 1024;  // LDS of a CU

template <class VT, class XT, class ACC>
struct TailLevel {
  ColIdx ci;
  ValSrc<VT, ACC> src;
  const uint8_t *dslot;
  const int *inj;    // the transfer to the next level
  const int *frow;
  const float *sigma;
  int ninj, row0;
  const int *boffs;  // the blocks' distances (has_block_offs) where sweep_slot takes the level, else null
  int npad, ncol;
  int xoff, roff;    // x (and a zero) and r in LDS, in elements
  int start[kTailColours + 1];
};
// r, x: the first level's.  load_x: start from x instead of 0.
template <class VT, class XT, class ACC>
struct TailArgs {
  TailLevel<VT, XT, ACC> lv[kMaxLevels];
  const XT *r;
  XT *x;
  int n, load_x;
};

template <class VT, class XT, class ACC, bool SCALE, int CF, int VF, bool GEN>
__global__ __launch_bounds__(kTailThreads) void k_tail(const TailArgs<VT, XT, ACC> a) {
  extern __shared__ double tail_shared[];
  XT *lds = reinterpret_cast<XT *>(tail_shared);
  const int lane = threadIdx.x & 63, nw = blockDim.x >> 6;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  // A sweep of a kValsSlot level whose blocks have one distance per slot, one
  // diagonal, and a slice or none for every wave.  A step then is LDS reads, a
  // chain of 27 sums, a division and a barrier: what comes from memory (the
  // row's mask) is fetched a step ahead, the slots' values and the level's
  // fields are read once.  A slot without an entry reads the zero that lies behind
  // the level's x.  (20^3: its second level has an odd size and takes the sweep
  // below.)
  auto sweep_slot = [&](const TailLevel<VT, XT, ACC> &L) {
    XT *x = lds + L.xoff;
    const XT *r = lds + L.roff;
    const int npad = L.npad, ncol = L.ncol, steps = 2 * ncol - 1;
    const int *boffs = L.boffs, *start = L.start;
    const uint32_t *mask = L.src.mask;
    ACC sv[kSlots];
#pragma unroll
    for (int s = 0; s < kSlots; ++s) sv[s] = L.src.slotv[s];
    int k = 0, at = start[0] + wave * kSlice;
    bool in = at < start[1];
    uint32_t m = in ? mask[at + lane] : 0;
    for (int step = 0; step < steps; ++step) {
      const int kn = step + 1 < ncol ? step + 1 : step + 1 < steps ? 2 * ncol - 3 - step : 0;
      const int an = start[kn] + wave * kSlice;
      const bool inn = an < start[kn + 1];
      const uint32_t mn = inn ? mask[an + lane] : 0;
      if (in) {
        const int *off = boffs + k * kMeta;
        const int row = at + lane;
        const ACC d = (m >> kDiagSlot) & 1u ? sv[kDiagSlot] : (ACC)1;
        const ACC xi = (ACC)x[row];
        ACC sum = (ACC)r[row];
#pragma unroll
        for (int s = 0; s < kSlots; ++s) {
          if (s == kDiagSlot) sum -= d * xi;
          else sum -= sv[s] * (ACC)x[npad + ((row + off[s] - npad) & -(int)((m >> s) & 1u))];
        }
        sum += xi * d;
        x[row] = (XT)(sum / d);
      }
      __syncthreads();
      k = kn;
      at = an;
      in = inn;
      m = mn;
    }
  };
  auto sweep = [&](const TailLevel<VT, XT, ACC> &L) {  // forward, then backward without the last block
    if constexpr (VF == kValsSlot) {
      if (L.boffs) return sweep_slot(L);
    }
    XT *x = lds + L.xoff;
    for (int step = 0; step < 2 * L.ncol - 1; ++step) {
      const int k = step < L.ncol ? step : 2 * L.ncol - 2 - step;
      const int end = L.start[k + 1] >> 6;
      for (int slice = (L.start[k] >> 6) + wave; slice < end; slice += nw) {
        const int row = slice * kSlice + lane;
        x[row] = gs_value<VT, XT, ACC, -1, false, CF, VF, GEN>(L.ci, L.src, lds + L.roff, x, row, L.dslot);
      }
      __syncthreads();
    }
  };
  const TailLevel<VT, XT, ACC> &F = a.lv[0];
  for (int i = threadIdx.x; i < F.npad; i += blockDim.x) {
    lds[F.xoff + i] = a.load_x ? a.x[i] : (XT)0;
    lds[F.roff + i] = a.r[i];
  }
  for (int l = threadIdx.x; l < a.n; l += blockDim.x) lds[a.lv[l].xoff + a.lv[l].npad] = (XT)0;
  for (int l = 1; l < a.n; ++l)
    for (int i = threadIdx.x; i < a.lv[l].npad; i += blockDim.x) lds[a.lv[l].xoff + i] = lds[a.lv[l].roff + i] = (XT)0;
  __syncthreads();
  for (int l = 0;; ++l) {
    const TailLevel<VT, XT, ACC> &L = a.lv[l];
    const XT *x = lds + L.xoff;
    sweep(L);
    if (l + 1 == a.n) break;
    // the next level's r: residual at the injected rows (k_restrict)
    for (int t0 = wave * kSlice; t0 < L.ninj; t0 += nw * kSlice) {
      const int t = t0 + lane;
      if (t >= L.ninj) continue;
      const int64_t row = L.frow ? L.frow[t] : L.row0 + t;
      const size_t b = ell_base(row);
      RowVals<VF, VT, ACC, false, kAllSlots> v;
      v.load(L.src, row);
      auto row_ax = [&](auto cm, const int *base) {
        constexpr int CM = decltype(cm)::value;
        ACC ax = 0;
#pragma unroll
        for (int s = 0; s < kSlots; ++s) {
          const int c = col_at<CM, false>(L.ci, row, base, b, s);
          ax += v.at(s, c) * (ACC)x[c];
        }
        return ax;
      };
      ACC ax;
      if constexpr (GEN) ax = with_cols<CF, false>(L.ci, slice_of<false>(row), row_ax);  // rows from a list
      else ax = with_cols<CF, true>(L.ci, slice_of<true>(row), row_ax);
      if constexpr (!GEN) mend_nan<false>(ax, FromZero{}, L.ci.cols, L.src.vals, x, row, kAllSlots);
      ACC res = (ACC)lds[L.roff + row] - ax;
      if (SCALE) res = res * (ACC)L.sigma[t];
      lds[a.lv[l + 1].roff + L.inj[t]] = (XT)res;
    }
    __syncthreads();
  }
  for (int l = a.n - 2; l >= 0; --l) {
    const TailLevel<VT, XT, ACC> &L = a.lv[l];
    for (int t = threadIdx.x; t < L.ninj; t += blockDim.x) {  // k_prolong
      const int row = L.frow ? L.frow[t] : L.row0 + t;
      ACC v = (ACC)lds[a.lv[l + 1].xoff + L.inj[t]];
      if (SCALE) v = v * (ACC)L.sigma[t];
      lds[L.xoff + row] = (XT)((ACC)lds[L.xoff + row] + v);
    }
    __syncthreads();
    sweep(L);
  }
  for (int i = threadIdx.x; i < F.npad; i += blockDim.x) a.x[i] = lds[F.xoff + i];
}

// ---------------------------------------------------------------------------
// element-wise helpers

// w = alpha x + beta y with the branches of ComputeWAXPBY_ref.cpp:52-67
__device__ __forceinline__ double waxpby1(double alpha, double x, double beta, double y) {
  if (alpha == 1.0) return x + beta * y;
  if (beta == 1.0) return alpha * x + y;
  return alpha * x + beta * y;
}

}  // namespace hpcgx
