// What the tile einsum kernels share: the pairs a launch walks, the mapping of
// blocks to XCDs and the geometry of a GEMM-shaped tile einsum.
#pragma once

#include "ej_internal.h"

namespace ej {

// ---------------------------------------------------------------------------
// Shared pair addressing.

struct PairSrc {
  const int64_t *lidx, *ridx;  // null: identity
  const int32_t *perm;         // null: identity
  const int32_t *seg_off;      // null: one pair per segment
  int64_t n_a_tiles, n_b_tiles;
  const int64_t *n_live;       // non-null: segments >= *n_live are skipped (grid is a bound)
  const int32_t *run_order;    // non-null: grouped launches run group run_order[b] as block b
  int32_t order_group;         // segments per group that run_order was made for
};

// Whether the workgroup's segment lies beyond the device-side segment count.
__device__ inline bool seg_dead(const PairSrc &s, int64_t seg) {
  return s.n_live && seg >= *s.n_live;
}

__device__ inline void seg_range(const PairSrc &s, int64_t seg, int64_t *q0, int64_t *q1) {
  if (s.seg_off) {
    *q0 = s.seg_off[seg];
    *q1 = s.seg_off[seg + 1];
  } else {
    *q0 = seg;
    *q1 = seg + 1;
  }
}

// Tiles of the q-th pair in plan order; false if an index is out of range.
__device__ inline bool pair_tiles(const PairSrc &s, int64_t q, int64_t *at, int64_t *bt) {
  int64_t p = s.perm ? s.perm[q] : q;
  *at = s.lidx ? s.lidx[p] : p;
  *bt = s.ridx ? s.ridx[p] : p;
  return *at >= 0 && *at < s.n_a_tiles && *bt >= 0 && *bt < s.n_b_tiles;
}

__device__ inline float to_f32(float x) { return x; }
__device__ inline float to_f32(uint16_t x) { return __uint_as_float(static_cast<uint32_t>(x) << 16); }

// Output element stores: fp32 as is, bf16 rounded to nearest even
// (v_cvt_pk_bf16_f32).  Sums are always formed in fp32; a bf16 output is
// rounded once, when the finished tile is written.
__device__ inline void put_out(float *p, float v) { *p = v; }
__device__ inline void put_out(uint16_t *p, float v) {
  *p = __builtin_bit_cast(uint16_t, static_cast<__bf16>(v));
}

// Reads a workgroup-uniform element of a read-only index array through the
// scalar cache, so the load does not occupy the vector memory counter that
// paces the LDS ring.
template <typename T>
__device__ inline T ld_uniform(const T *p, int64_t i) {
  return ((const __attribute__((address_space(4))) T *)(p))[i];
}

// Maps the first `live` block ids onto logical blocks (block id b runs on XCD
// b % 8).  run == 0: the logical range is split into 8 contiguous parts, one
// per XCD, so that neighbouring logical blocks (sharing operand tiles) share
// an L2 over the widest window.  run > 0: runs of `run` consecutive logical
// blocks go to one XCD, the runs dealt to the XCDs in turn, so that every XCD
// gets a share of each region of the logical range (work that is heavier in
// one region, as for skewed sparsity, stays balanced); the last, partial
// round of runs is split into 8 contiguous parts.  Block ids from `live` on
// keep their id: they lie beyond the work of a grid sized for a bound.
__device__ inline uint32_t xcd_logical_block(uint32_t live, uint32_t run = 0) {
  const uint32_t bid = blockIdx.x;
  if (bid >= live) return bid;
  const uint32_t full = run > 0 ? live / (8 * run) * (8 * run) : 0;
  const uint32_t xcd = bid % 8;
  if (bid < full) {
    const uint32_t local = bid / 8;
    return ((local / run) * 8 + xcd) * run + local % run;
  }
  const uint32_t rest = live - full, local = (bid - full) / 8;
  const uint32_t per = rest / 8, rem = rest % 8;
  const uint32_t start = xcd < rem ? xcd * (per + 1) : rem * (per + 1) + (xcd - rem) * per;
  return full + start + local;
}

// x / d (and the remainder) of workgroup-uniform values, kept in scalar
// registers.  A division runs on the vector unit (a 64-bit one takes over a
// hundred instructions), and what follows from its result would stay there:
// one division of 1 is the common case and costs nothing.
__device__ inline uint32_t div_uniform(uint32_t x, uint32_t d, uint32_t *rem) {
  if (d == 1) {
    *rem = 0;
    return x;
  }
  const uint32_t q = __builtin_amdgcn_readfirstlane(x / d);
  *rem = x - q * d;
  return q;
}

// Run length of the dealt mapping for one-segment workgroups taken in plan
// order (no run order): their neighbours share few tiles, and skewed
// sparsity makes whole regions of the plan heavier.
constexpr uint32_t kXcdRun = 16;

// Blocks that carry work when each segment takes blocks_per_seg of them: the
// whole grid, or, given a device-side segment count, that many segments' blocks
// (so that a grid sized for a bound still spreads its live work over every XCD).
__device__ inline uint32_t live_blocks(const PairSrc &s, int64_t blocks_per_seg) {
  const uint32_t total = gridDim.x;
  if (!s.n_live) return total;
  const int64_t live = ld_uniform(s.n_live, 0) * blocks_per_seg;
  return live < total ? static_cast<uint32_t>(live) : total;
}

// ---------------------------------------------------------------------------
// GEMM-shaped tile einsums.

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

struct GemmGeom {
  int64_t m, n, k, batch;
  int64_t a_sb, a_sm, a_sk, b_sb, b_sk, b_sn, c_sb, c_sm, c_sn;
  int64_t a_elems, b_elems, c_elems;
  int64_t mblocks, nblocks;
  int32_t out_bf16;  // output tiles in bf16 (else fp32)
};

// Where an output block lies: n-block, m-block, batch index, segment (or
// group of segments) of logical block lb.
struct BlockPos {
  uint32_t nb, mb, bi, seg;
};
__device__ inline BlockPos block_pos(uint32_t lb, const GemmGeom &g, bool all_m = false) {
  BlockPos p{0, 0, 0, 0};
  lb = div_uniform(lb, static_cast<uint32_t>(g.nblocks), &p.nb);
  if (!all_m) lb = div_uniform(lb, static_cast<uint32_t>(g.mblocks), &p.mb);
  p.seg = div_uniform(lb, static_cast<uint32_t>(g.batch), &p.bi);
  return p;
}

}  // namespace ej
