// Streaming tile GEMM: operands go from memory straight into the MFMA's
// registers, for any tile extents, strides and alignment.
//
// The LDS-ring kernels need extents that are multiples of their blocks and
// 16-byte rows.  Tile extents are divisors of the data's extents, so odd ones
// are ordinary; those ran one thread per output element.  Here a wave holds a
// block of FM x FN MFMA fragments (16 x 16 each, up to 5 x 5) of one output
// tile and walks "K blocks" (16 deep for fp32, 32 for bf16) of the segment's
// pairs, loading each lane's fragment values itself:
//   KC  the contraction dimension is contiguous: a lane's k values of one row
//       are 16 consecutive bytes, one load (2- or 4-byte aligned; the
//       hardware takes unaligned vector loads).
//   FC  the free dimension is contiguous: the MFMA's 16 columns are free to
//       stand for any 16 columns as long as the result is stored under the
//       same names, so lane q takes columns w q .. w q + w - 1 of a group of w
//       fragments (w = 4, 2, 1) and one load of w elements per k row feeds
//       w fragments.  The results of a group then lie in w consecutive
//       columns per lane and leave with one store.
//   GS  neither: one element per load.
// Rows and columns past the tile's edge are clamped onto the last valid ones
// (KC, GS: not stored; FC: the whole group moves back, so lanes write
// the same values twice).  k past the end is zeroed in both operands, so
// nothing outside a tile is ever read and an Inf or NaN in the tile meets
// only its own products.
// W waves share a segment: wave w takes K blocks w, w + W, ... of the
// segment's whole run of pairs, so the waves are balanced for every number of
// fragments and of pairs, need no barrier while they stream, and add their
// blocks once at the end through LDS, in wave order.  W = 4 where there are
// too few output blocks to fill the chip, W = 1 (four output blocks to a
// workgroup, LDS unused) otherwise.  The two add a segment's K blocks in
// different orders, so the choice is made on the device from the segments
// that are there, never from the bound a launch is sized for: an einsum then
// gives the same bits whether its plan was counted first or queued.
// Measured (one MI355X), against one thread per output element: block-sparse
// 6000^2 x dense 6000 x 1500 fp32, 75 x 75 tiles (12,800 pairs, 10.8 GFLOP)
// 170 us / 3,380 us: 64 TFLOP/s, fp32 MFMAs 47% busy (two workgroups fit a CU, so
// the 1,600 run as three full rounds of 512 and an eighth of a fourth).  Sparse x
// sparse 10240^2 bf16, 80 x 80 tiles (5,240 pairs) 32 us / 1,750 us, bound by the
// latency of a pair's three K blocks, the only ones of most segments.
#pragma once

#include <algorithm>

#include "ej_gemm.h"

namespace ej {

enum StreamMode { kStreamKC = 0, kStreamFC = 1, kStreamGS = 2 };

typedef int i32x2s_t __attribute__((ext_vector_type(2)));
typedef int i32x4s_t __attribute__((ext_vector_type(4)));
typedef float f32x2s_t __attribute__((ext_vector_type(2)));
// Vectors at element alignment.
typedef i32x4s_t i32x4_u2 __attribute__((aligned(2)));
typedef i32x2s_t i32x2_u2 __attribute__((aligned(2)));
typedef int i32_u2 __attribute__((aligned(2)));
typedef i32x4s_t i32x4_u4 __attribute__((aligned(4)));
typedef i32x2s_t i32x2_u4 __attribute__((aligned(4)));

// 16 bytes at base + off.
template <typename T>
__device__ inline i32x4s_t stream_ld16(const T *base, uint32_t off) {
  if constexpr (sizeof(T) == 2) return *reinterpret_cast<const i32x4_u2 *>(base + off);
  else return *reinterpret_cast<const i32x4_u4 *>(base + off);
}

// One operand of a wave: F fragments of its free dimension.
template <typename T, int F, int MODE>
struct StreamOp {
  static constexpr bool BF = sizeof(T) == 2;
  static constexpr int KL = BF ? 8 : 4;  // k values per lane and K block
  static constexpr int KB = 4 * KL;
  // FC groups: fragments 0 .. 3 as one group of four, then a pair, then a
  // single one.
  static constexpr int G4 = MODE == kStreamFC ? F / 4 : 0;
  static constexpr int G2 = MODE == kStreamFC ? F % 4 / 2 : 0;
  static constexpr int G1 = MODE == kStreamFC ? F % 2 : 0;
  static_assert(F >= 1 && F <= 7, "fragments per operand");
  static constexpr int NOFF = MODE == kStreamFC ? G4 + G2 + G1 : F;
  // A loaded K block, in the vectors the loads wrote (moving their elements
  // apart here would wait for the loads).
  static constexpr int N4 = MODE == kStreamKC ? F : MODE == kStreamFC && !BF ? 4 * G4 : 0;
  static constexpr int N2 = MODE == kStreamFC ? (BF ? 8 * G4 : 4 * G2) : 0;
  static constexpr int N1 = MODE == kStreamGS ? KL * F
                            : MODE == kStreamFC ? (BF ? 8 * (G2 + G1) : 4 * G1)
                                                : 0;
  struct Raw {
    i32x4s_t v4[N4 ? N4 : 1];
    i32x2s_t v2[N2 ? N2 : 1];
    int v1[N1 ? N1 : 1];
  };
  uint32_t off[NOFF];  // free-dimension offset of each fragment or group
  uint32_t lane_k;     // KC: first k of this lane; else its offset KL g s_k

  // Index along the free dimension of result row / column `idx` (0 .. 15) of
  // fragment f, for a block that starts at `first` of `ext`.
  __device__ static int free_index(int f, int idx, int first, int ext) {
    if constexpr (MODE == kStreamFC) {
      const int f0 = f < 4 * G4 ? 0 : f < 4 * G4 + 2 * G2 ? 4 * G4 : 4 * G4 + 2 * G2;
      const int w = f < 4 * G4 ? 4 : f < 4 * G4 + 2 * G2 ? 2 : 1;
      const int s = first + 16 * f0 + w * idx;
      return (s < ext - w ? s : ext - w) + (f - f0);
    } else {
      return first + 16 * f + idx;
    }
  }

  __device__ void init(int lane, int first, int ext, uint32_t s_free, uint32_t s_k) {
    const int q = lane & 15, g = lane >> 4;
    lane_k = MODE == kStreamKC ? KL * g : KL * g * s_k;
    if constexpr (MODE == kStreamFC) {
#pragma unroll
      for (int t = 0; t < NOFF; ++t) {
        const int f0 = t < G4 ? 4 * t : 4 * G4 + 2 * (t - G4);
        off[t] = static_cast<uint32_t>(free_index(f0, q, first, ext));
      }
    } else {
#pragma unroll
      for (int i = 0; i < F; ++i) {
        int r = first + 16 * i + q;
        r = r < ext ? r : ext - 1;
        off[i] = r * s_free;
      }
    }
  }

  // Loads K block k0 of the tile at `base` (uniform).  A KC lane whose k
  // values reach past K loads the last KL of its row instead (pack moves them
  // into place); FC and GS rows past K are the last row (pack zeroes them).
  __device__ void load(const T *base, uint32_t k0, uint32_t K, uint32_t s_k, Raw &raw) const {
    if constexpr (MODE == kStreamKC) {
      uint32_t k = k0 + lane_k;
      k = k < K - KL ? k : K - KL;
#pragma unroll
      for (int i = 0; i < F; ++i) raw.v4[i] = stream_ld16(base, off[i] + k);
    } else {
      const uint32_t x0 = k0 * s_k + lane_k, last = (K - 1) * s_k;
#pragma unroll
      for (int kk = 0; kk < KL; ++kk) {
        uint32_t x = x0 + kk * s_k;
        x = x < last ? x : last;
        int i4 = 0, i2 = 0, i1 = 0;
#pragma unroll
        for (int t = 0; t < NOFF; ++t) {
          const T *e = base;
          const uint32_t y = off[t] + x;
          if constexpr (MODE == kStreamGS) {
            raw.v1[KL * t + kk] = BF ? static_cast<int>(e[y]) : __float_as_int(to_f32(e[y]));
          } else if (t < G4) {
            if constexpr (BF) raw.v2[8 * i2 + kk] = *reinterpret_cast<const i32x2_u2 *>(e + y);
            else raw.v4[4 * i4 + kk] = *reinterpret_cast<const i32x4_u4 *>(e + y);
            ++i2;
            ++i4;
          } else if (t < G4 + G2) {
            if constexpr (BF) {
              raw.v1[8 * i1 + kk] = *reinterpret_cast<const i32_u2 *>(e + y);
              ++i1;
            } else {
              raw.v2[kk] = *reinterpret_cast<const i32x2_u4 *>(e + y);
            }
          } else {
            if constexpr (BF) raw.v1[8 * i1 + kk] = static_cast<int>(e[y]);
            else raw.v1[kk] = __float_as_int(to_f32(e[y]));
          }
        }
      }
    }
  }

  // Dword x of the lane's 16 bytes of fragment f (fp32: k = x; bf16: k = 2x
  // low, 2x + 1 high).
  __device__ static int dword(const Raw &raw, int f, int x) {
    if constexpr (MODE == kStreamKC) {
      return raw.v4[f][x];
    } else if constexpr (!BF) {
      if constexpr (MODE == kStreamGS) return raw.v1[4 * f + x];
      else if (f < 4 * G4) return raw.v4[x][f];
      else if (f < 4 * G4 + 2 * G2) return raw.v2[x][f - 4 * G4];
      else return raw.v1[x];
    } else {
      auto lo2 = [](int a, int b) {
        return static_cast<int>(__builtin_amdgcn_perm(b, a, 0x05040100u));
      };
      auto hi2 = [](int a, int b) {
        return static_cast<int>(__builtin_amdgcn_perm(b, a, 0x07060302u));
      };
      if constexpr (MODE == kStreamGS) {
        return lo2(raw.v1[8 * f + 2 * x], raw.v1[8 * f + 2 * x + 1]);
      } else if (f < 4 * G4) {
        const int a = raw.v2[2 * x][f >> 1 & 1], b = raw.v2[2 * x + 1][f >> 1 & 1];
        return f & 1 ? hi2(a, b) : lo2(a, b);
      } else if (f < 4 * G4 + 2 * G2) {
        return (f - 4 * G4) & 1 ? hi2(raw.v1[2 * x], raw.v1[2 * x + 1])
                                : lo2(raw.v1[2 * x], raw.v1[2 * x + 1]);
      } else {
        return lo2(raw.v1[8 * G2 + 2 * x], raw.v1[8 * G2 + 2 * x + 1]);
      }
    }
  }

  // The fragments of a loaded K block, k past K zeroed.
  __device__ void pack(const Raw &raw, uint32_t k0, uint32_t K, int lane,
                       i32x4s_t (&fr)[F]) const {
#pragma unroll
    for (int f = 0; f < F; ++f)
#pragma unroll
      for (int x = 0; x < 4; ++x) fr[f][x] = dword(raw, f, x);
    if (k0 + KB <= K) return;  // uniform
    const int over = static_cast<int>(k0 + KL * (lane >> 4)) - static_cast<int>(K - KL);
    if constexpr (MODE == kStreamKC) {
      // the values were loaded `over` elements early: shift them down
      const int s = over > 0 ? over : 0;
      const int ds = BF ? s >> 1 : s;
#pragma unroll
      for (int f = 0; f < F; ++f) {
        int x[5];
#pragma unroll
        for (int d = 0; d < 4; ++d) {
          int v = 0;
#pragma unroll
          for (int e = 3; e >= d; --e) v = ds == e - d ? fr[f][e] : v;
          x[d] = v;
        }
        x[4] = 0;
#pragma unroll
        for (int d = 0; d < 4; ++d)
          fr[f][d] = BF && (s & 1) ? static_cast<int>(__builtin_amdgcn_alignbit(x[d + 1], x[d], 16))
                                   : x[d];
      }
    } else {
      const int n = KL - over;  // valid k values of this lane
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        const int m = !BF ? (x < n ? -1 : 0) : n >= 2 * x + 2 ? -1 : n == 2 * x + 1 ? 0xFFFF : 0;
#pragma unroll
        for (int f = 0; f < F; ++f) fr[f][x] &= m;
      }
    }
  }
};

// Vector stores of a group's w consecutive results (element aligned).
template <int N>
__device__ inline void stream_put(float *p, const float *v) {
  if constexpr (N == 4)
    *reinterpret_cast<i32x4_u4 *>(p) =
        i32x4s_t{__float_as_int(v[0]), __float_as_int(v[1]), __float_as_int(v[2]),
                 __float_as_int(v[3])};
  else if constexpr (N == 2)
    *reinterpret_cast<i32x2_u4 *>(p) = i32x2s_t{__float_as_int(v[0]), __float_as_int(v[1])};
  else *p = v[0];
}
template <int N>
__device__ inline void stream_put(uint16_t *p, const float *v) {
  uint16_t h[4];
#pragma unroll
  for (int i = 0; i < N; ++i) put_out(&h[i], v[i]);
  if constexpr (N == 4)
    *reinterpret_cast<i32x2_u2 *>(p) =
        i32x2s_t{h[0] | (h[1] << 16), h[2] | (h[3] << 16)};
  else if constexpr (N == 2)
    *reinterpret_cast<i32_u2 *>(p) = h[0] | (h[1] << 16);
  else *p = h[0];
}

// Registers of a wave: 4 FM FN accumulators, two sets of raw operands and the
// packed fragments.  Large blocks get two waves per SIMD, small ones more.
constexpr int stream_waves(int nf) { return nf >= 15 ? 2 : nf >= 9 || nf == 5 ? 3 : 4; }

// Below this many output blocks four waves share each.  2048 is the chip's
// wave slots at two waves per SIMD: fewer blocks cannot fill it one wave each.
// Measured, one wave / four waves a block: 80 x 80 bf16, ~4,500 blocks of 1.2
// pairs 32 / 73 us (most of a split block's time is its reduction); 120 x 120
// bf16, 4,592 blocks 25 / 31 us; 75 x 75 fp32, 1,600 blocks of 8 pairs 219 /
// 170 us; 36 x 36 fp32, 252 blocks of up to 50 pairs 58 / 19 us.
constexpr int64_t kStreamSplitBlocks = 2048;

// Output block lb (uniform over the wave) of the launch; `part`: the W = 4
// reduction's LDS.  Every wave of a W = 4 workgroup calls it with one lb.
template <typename T, int FM, int FN, int AMODE, int BMODE, int W>
__device__ inline void stream_block(const T *__restrict__ A, const T *__restrict__ B,
                                    void *__restrict__ C, const PairSrc &src, const GemmGeom &g,
                                    uint32_t lb, float *part) {
#if defined(__HIP_DEVICE_COMPILE__)
  using OA = StreamOp<T, FM, AMODE>;
  using OB = StreamOp<T, FN, BMODE>;
  constexpr bool BF = OA::BF;
  constexpr int KB = OA::KB;
  constexpr int NF = FM * FN;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const BlockPos at_block = block_pos(lb, g);
  const int nb = static_cast<int>(at_block.nb), mb = static_cast<int>(at_block.mb);
  const int64_t bi = at_block.bi, seg = at_block.seg;
  const int32_t q0 = src.seg_off ? ld_uniform(src.seg_off, seg) : static_cast<int32_t>(seg);
  const int32_t q1 = src.seg_off ? ld_uniform(src.seg_off, seg + 1) : q0 + 1;
  const int M = static_cast<int>(g.m), N = static_cast<int>(g.n), K = static_cast<int>(g.k);
  const int m0 = mb * FM * 16, n0 = nb * FN * 16;
  const int kbp = (K + KB - 1) / KB;  // K blocks per pair
  const uint32_t ask = static_cast<uint32_t>(g.a_sk), bsk = static_cast<uint32_t>(g.b_sk);
  OA oa;
  OB ob;
  oa.init(lane, m0, M, static_cast<uint32_t>(g.a_sm), ask);
  ob.init(lane, n0, N, static_cast<uint32_t>(g.b_sn), bsk);
  const T *const a0 = A + bi * g.a_sb;
  const T *const b0 = B + bi * g.b_sb;

  // The segment's pairs, one per lane, 64 at a time (-1: an index out of
  // range, whose products are left out).
  int32_t ta = -1, tb = -1;
  int chunk = -1;
  const int32_t len = q1 - q0;
  auto load_table = [&](int c) {
    const int r = c * 64 + lane;
    int32_t na = -1, nb_ = -1;
    if (r < len) {
      const int64_t q = static_cast<int64_t>(q0) + r;
      const int64_t p = src.perm ? src.perm[q] : q;
      const int64_t a = src.lidx ? src.lidx[p] : p;
      const int64_t b = src.ridx ? src.ridx[p] : p;
      const bool ok = a >= 0 && a < src.n_a_tiles && b >= 0 && b < src.n_b_tiles;
      na = ok ? static_cast<int32_t>(a) : -1;
      nb_ = ok ? static_cast<int32_t>(b) : -1;
    }
    ta = na;
    tb = nb_;
    chunk = c;
  };

  f32x4_t acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  // K blocks of this wave: s = w, w + W, ... of len * kbp.
  const int w0 = W == 1 ? 0 : wave;
  const int64_t total = static_cast<int64_t>(len) * kbp;
  const int64_t mine = total > w0 ? (total - w0 + W - 1) / W : 0;
  if (mine > 0) {
    int pos = 0, kc = w0;  // cursor of the next K block to load
    while (kc >= kbp) { kc -= kbp; ++pos; }
    typename OA::Raw raw_a[2];
    typename OB::Raw raw_b[2];
    uint32_t k0s[2];  // K block of each set
    bool okp[2];      // its pair's indices are valid
    int64_t left = mine;
    // Loads the next K block into a set and moves the cursor.  After the last
    // one it loads that one again: the number of loads in flight then does
    // not depend on a branch, and each wait stays exact.
    auto issue = [&](int set) {
      if ((pos >> 6) != chunk) load_table(pos >> 6);
      const int32_t at = __builtin_amdgcn_readlane(ta, pos & 63);
      const int32_t bt = __builtin_amdgcn_readlane(tb, pos & 63);
      const int64_t a_tile = at < 0 ? 0 : at, b_tile = bt < 0 ? 0 : bt;
      const uint32_t k0 = kc * KB;
      oa.load(a0 + a_tile * g.a_elems, k0, K, ask, raw_a[set]);
      ob.load(b0 + b_tile * g.b_elems, k0, K, bsk, raw_b[set]);
      k0s[set] = k0;
      okp[set] = at >= 0;
      if (--left > 0) {
        kc += W;
        while (kc >= kbp) { kc -= kbp; ++pos; }
      }
    };
    auto compute = [&](int set) {
      if (!okp[set]) return;
      i32x4s_t fa[FM], fb[FN];
      oa.pack(raw_a[set], k0s[set], K, lane, fa);
      ob.pack(raw_b[set], k0s[set], K, lane, fb);
      if constexpr (BF) {
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
          for (int j = 0; j < FN; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                __builtin_bit_cast(bf16x8_t, fa[i]), __builtin_bit_cast(bf16x8_t, fb[j]),
                acc[i][j], 0, 0, 0);
      } else {
        // A K block's 16 products are summed apart and added to the block's
        // total: sums of long segments then lose less than one running chain.
#pragma unroll
        for (int i = 0; i < FM; ++i) {
          f32x4_t t[FN];
#pragma unroll
          for (int c = 0; c < 4; ++c)
#pragma unroll
            for (int j = 0; j < FN; ++j)
              t[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                  __int_as_float(fa[i][c]), __int_as_float(fb[j][c]),
                  c == 0 ? f32x4_t{0.f, 0.f, 0.f, 0.f} : t[j], 0, 0, 0);
#pragma unroll
          for (int j = 0; j < FN; ++j) acc[i][j] += t[j];
        }
      }
    };
    // Two K blocks a round, with no branch between a set's loads and its use.
    issue(0);
    for (int64_t t = mine >> 1; t != 0; --t) {
      issue(1);
      compute(0);
      issue(0);
      compute(1);
    }
    if (mine & 1) compute(0);
  }

  const int q = lane & 15, gq = lane >> 4;
  const int64_t c0 = seg * g.c_elems + bi * g.c_sb;
  const int64_t csm = g.c_sm, csn = g.c_sn;
  // One row (result row 4 gq + r of fragment i) of this wave's block.
  auto put_row = [&](auto *cb, int i, int r, const float (&v)[FN]) {
    const int m = OA::free_index(i, 4 * gq + r, m0, M);
    if (AMODE != kStreamFC && m >= M) return;
    auto *row = cb + static_cast<int64_t>(m) * csm;
    if (BMODE == kStreamFC && csn == 1) {
#pragma unroll
      for (int t = 0; t < OB::NOFF; ++t) {
        const int f0 = t < OB::G4 ? 4 * t : 4 * OB::G4 + 2 * (t - OB::G4);
        const int n = OB::free_index(f0, q, n0, N);
        if (t < OB::G4) stream_put<4>(row + n, v + f0);
        else if (t < OB::G4 + OB::G2) stream_put<2>(row + n, v + f0);
        else stream_put<1>(row + n, v + f0);
      }
    } else {
#pragma unroll
      for (int j = 0; j < FN; ++j) {
        const int n = OB::free_index(j, q, n0, N);
        if (n < N) put_out(row + n * csn, v[j]);
      }
    }
  };
  if constexpr (W == 1) {
    auto store = [&](auto *cb) {
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          float v[FN];
#pragma unroll
          for (int j = 0; j < FN; ++j) v[j] = acc[i][j][r];
          put_row(cb, i, r, v);
        }
    };
    if (g.out_bf16) store(static_cast<uint16_t *>(C) + c0);
    else store(static_cast<float *>(C) + c0);
  } else {
    // Wave r sums and stores result rows 4 gq + r of every fragment: each wave
    // hands the other three their rows through LDS (one float per lane and
    // fragment, consecutive lanes on consecutive banks).
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      if (r == wave) continue;
      float *dst = part + static_cast<size_t>((r * 3 + (wave < r ? wave : wave - 1)) * NF) * 64 + lane;
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) dst[(i * FN + j) * 64] = acc[i][j][r];
    }
    __syncthreads();
    auto store = [&](auto *cb) {
#pragma unroll
      for (int i = 0; i < FM; ++i) {
        float v[FN];
#pragma unroll
        for (int j = 0; j < FN; ++j) {
          const float own = wave == 0 ? acc[i][j][0] : wave == 1 ? acc[i][j][1]
                            : wave == 2 ? acc[i][j][2] : acc[i][j][3];
          float s = 0.f;
#pragma unroll
          for (int w = 0; w < 4; ++w) {
            const int slot = w < wave ? w : w - 1;
            const float x = w == wave
                                ? own
                                : part[((wave * 3 + slot) * NF + i * FN + j) * 64 + lane];
            s = w == 0 ? x : s + x;
          }
          v[j] = s;
        }
        put_row(cb, i, wave, v);
      }
    };
    if (g.out_bf16) store(static_cast<uint16_t *>(C) + c0);
    else store(static_cast<float *>(C) + c0);
  }
#endif
}

template <typename T, int FM, int FN, int AMODE, int BMODE>
__global__ __launch_bounds__(256, stream_waves(FM * FN)) void stream_gemm_kernel(
    const T *__restrict__ A, const T *__restrict__ B, void *__restrict__ C, PairSrc src, GemmGeom g,
    int64_t n_seg) {
#if defined(__HIP_DEVICE_COMPILE__)
  __shared__ float part[4 * 3 * FM * FN * 64];
  int64_t nseg = n_seg;
  if (src.n_live) {
    const int64_t nl = ld_uniform(src.n_live, 0);
    nseg = nl < nseg ? nl : nseg;
  }
  // below 2^26 (try_stream)
  const uint32_t units = static_cast<uint32_t>(nseg * (g.nblocks * g.mblocks * g.batch));
  if (units < kStreamSplitBlocks) {
    if (blockIdx.x >= units) return;
    stream_block<T, FM, FN, AMODE, BMODE, 4>(A, B, C, src, g, xcd_logical_block(units, kXcdRun),
                                             part);
  } else {
    const uint32_t live = (units + 3) / 4;
    if (blockIdx.x >= live) return;
    const uint32_t lb = xcd_logical_block(live, kXcdRun) * 4 +
                        __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (lb >= units) return;
    stream_block<T, FM, FN, AMODE, BMODE, 1>(A, B, C, src, g, lb, part);
  }
#endif
}

// Fragments per wave along an extent: the extent's fragments split evenly
// over the fewest blocks of at most five.
inline int stream_frags(int64_t ext) {
  const int64_t f = ceil_div(ext, 16);
  return static_cast<int>(ceil_div(f, ceil_div(f, 5)));
}

// Launches the streaming GEMM (g.mblocks, g.nblocks are set here).
int launch_stream_f32(int amode, int bmode, const void *A, const void *B, void *C,
                      const PairSrc &src, GemmGeom g, int64_t n_seg, hipStream_t stream);
int launch_stream_bf16(int amode, int bmode, const void *A, const void *B, void *C,
                       const PairSrc &src, GemmGeom g, int64_t n_seg, hipStream_t stream);

template <typename T, int FM, int FN, int AMODE, int BMODE>
int launch_stream_t(const void *A, const void *B, void *C, const PairSrc &src, GemmGeom g,
                    int64_t n_seg, hipStream_t stream) {
  g.mblocks = ceil_div(g.m, FM * 16);
  g.nblocks = ceil_div(g.n, FN * 16);
  // One workgroup per output block below the split, one per four from it on; a
  // bound's live blocks may fall on either side.
  const int64_t units = n_seg * g.mblocks * g.nblocks * g.batch;
  int64_t nblk = units < kStreamSplitBlocks ? units : ceil_div(units, 4);
  if (src.n_live && units >= kStreamSplitBlocks) nblk = std::max(nblk, kStreamSplitBlocks - 1);
  hipLaunchKernelGGL((stream_gemm_kernel<T, FM, FN, AMODE, BMODE>),
                     dim3(static_cast<unsigned>(nblk)), dim3(256), 0, stream,
                     static_cast<const T *>(A), static_cast<const T *>(B), C, src, g, n_seg);
  EJ_LAUNCH_CHECK();
  return EJ_OK;
}

template <typename T, int AMODE, int BMODE, int FM>
int launch_stream_n(int fn, const void *A, const void *B, void *C, const PairSrc &src,
                    const GemmGeom &g, int64_t n_seg, hipStream_t stream) {
  switch (fn) {
    case 1: return launch_stream_t<T, FM, 1, AMODE, BMODE>(A, B, C, src, g, n_seg, stream);
    case 2: return launch_stream_t<T, FM, 2, AMODE, BMODE>(A, B, C, src, g, n_seg, stream);
    case 3: return launch_stream_t<T, FM, 3, AMODE, BMODE>(A, B, C, src, g, n_seg, stream);
    case 4: return launch_stream_t<T, FM, 4, AMODE, BMODE>(A, B, C, src, g, n_seg, stream);
    default: return launch_stream_t<T, FM, 5, AMODE, BMODE>(A, B, C, src, g, n_seg, stream);
  }
}

template <typename T, int AMODE, int BMODE>
int launch_stream_m(const void *A, const void *B, void *C, const PairSrc &src, const GemmGeom &g,
                    int64_t n_seg, hipStream_t stream) {
  const int fn = stream_frags(g.n);
  switch (stream_frags(g.m)) {
    case 1: return launch_stream_n<T, AMODE, BMODE, 1>(fn, A, B, C, src, g, n_seg, stream);
    case 2: return launch_stream_n<T, AMODE, BMODE, 2>(fn, A, B, C, src, g, n_seg, stream);
    case 3: return launch_stream_n<T, AMODE, BMODE, 3>(fn, A, B, C, src, g, n_seg, stream);
    case 4: return launch_stream_n<T, AMODE, BMODE, 4>(fn, A, B, C, src, g, n_seg, stream);
    default: return launch_stream_n<T, AMODE, BMODE, 5>(fn, A, B, C, src, g, n_seg, stream);
  }
}

// Strides that are contiguous in neither dimension (or an [k][m] lhs with an
// [n][k] rhs) run element loads on a few block shapes.
template <typename T>
int launch_stream_gs(const void *A, const void *B, void *C, const PairSrc &src, const GemmGeom &g,
                     int64_t n_seg, hipStream_t stream) {
  const int f = g.m > g.n ? stream_frags(g.m) : stream_frags(g.n);
  if (f <= 1)
    return launch_stream_t<T, 1, 1, kStreamGS, kStreamGS>(A, B, C, src, g, n_seg, stream);
  return launch_stream_t<T, 2, 2, kStreamGS, kStreamGS>(A, B, C, src, g, n_seg, stream);
}

}  // namespace ej
