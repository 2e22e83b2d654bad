// Tiled cost-volume kernels for gfx950 (MEAN and MIN / MAX reduces, every op of the family).
//
// Work decomposition.  A workgroup is one wavefront.  It owns PPW = 64/LPP pixels of one
// image (a compact block, see tile_rows: its samples change their texel cell together more
// often than a long row's) and one contiguous segment of the D depth hypotheses; the LPP lanes
// of a pixel each own VEC consecutive channels (C = LPP*VEC), so every tap read and every
// cost-row write of a pixel is one contiguous C*sizeof(S) segment.  Depth runs innermost:
// along the walk the sample point of a view slides along an epipolar line by a fraction of
// a texel per step, so the four bilinear taps of the current texel cell stay in registers
// and are reloaded only when the cell changes.
//
// Each chunk of LPP depths is processed in two phases:
//   phase 1  lane (pixel p, j) reprojects depth d0+j of pixel p into every view (the
//            bit-exact code of warp.h), writes the valid-view count and leaves a small
//            record per (view, depth, pixel) in LDS: tap offset (or -1) and four weights
//            (backward: also the cell key and four depth-derivative weights);
//   phase 2  lane (pixel p, channel slice) walks the LPP depths, reading the records as
//            LDS broadcasts, and does the channel arithmetic with explicit fused
//            multiply-adds.
// With LPP == 1 a lane owns its whole pixel and the records stay in registers.
//
// Backward keeps, per view, a register image of the source-gradient contributions to the
// current cell.  When the cell changes the image is added into a per-view LDS
// window of ROWS x COLS texels that follows the wave's samples along the epipolar lines;
// neighbouring pixels hit the same texels, so most of the scatter is absorbed there.  A
// texel reaches memory when the window moves off it, as part of a dense run of
// global_atomic_add_f32.  ref_grad and the base-plane gradient are pixel-owned and
// accumulate in registers; they are stored once (one depth segment) or added once per
// segment.
#pragma once

#include <type_traits>

#include "internal.h"

namespace chop {
namespace tiled {

// Rows of a wave's pixel tile (PPW = 64 / LPP pixels, tile_rows x PPW / tile_rows): as square
// as the pixel count allows.  The samples of a compact tile cross texel boundaries at more
// nearly the same depths than those of a long row, so fewer wave iterations carry a cell
// change (MVSNet-stage workload, 8 pixels: 0.49 of them for 2 x 4 against 0.61 for 1 x 8;
// f16 cascade workload, 16 pixels: 0.49-0.68 per view for 4 x 4 against 0.57-0.75 for 2 x 8),
// and its footprint in the source image has fewer texels per pixel.
// `tall`: eight pixels as 4 x 2.
constexpr int tile_rows(int ppw, bool tall = false) {
  return ppw >= 64 ? 8 : ppw >= 16 || tall ? 4 : ppw >= 2 ? 2 : 1;
}

// A forward launch gives each XCD one band of tiles: the segments of a tile one after the other
// (kBands), or all first segments of the band, then all second ones (kBandsBySegment).
constexpr int kBands = -1, kBandsBySegment = -2;

struct Geometry {
  int hw;                  // H*W
  int tiles_per_image;     // ceil(hw / PPW)
  int nseg;                // depth segments
  int ngroups;             // view groups (backward only): workgroups that split the views
  int vper;                // views per group
  int seg;                 // depths per segment, multiple of LPP
  int64_t total_units;     // B * tiles_per_image * nseg * ngroups
  unsigned units_per_seg;  // B * tiles_per_image * ngroups
  int64_t units_per_xcd;   // kBands: ceil(total_units / 8); kBandsBySegment: ceil(units_per_seg / 8)
  int xcd_shift;           // log2 of the units dealt to one XCD at a time, or kBands, kBandsBySegment
  int64_t grid;            // workgroups to launch
  int tiles_x;             // tiles per image row (a tile: tile_rows(PPW) rows of pixels)
  int sub;                 // channels per correlation group (1 for squared difference)
  bool stream_halves;      // forward: rows that leave as half lines (half_lines) bypass the caches
  float src_h_max, src_w_max;  // (float)(srcH - 1), (float)(srcW - 1): acceptance bounds
};

// ---- vector access ---------------------------------------------------------------------
template <typename S>
__device__ __forceinline__ void widen_word(uint32_t w, float *out);
template <>
__device__ __forceinline__ void widen_word<float>(uint32_t w, float *out) {
  out[0] = __uint_as_float(w);
}
template <>
__device__ __forceinline__ void widen_word<__half>(uint32_t w, float *out) {
  out[0] = __half2float(__ushort_as_half((unsigned short)(w & 0xffffu)));
  out[1] = __half2float(__ushort_as_half((unsigned short)(w >> 16)));
}
template <>
__device__ __forceinline__ void widen_word<bf16_t>(uint32_t w, float *out) {
  out[0] = __uint_as_float(w << 16);
  out[1] = __uint_as_float(w & 0xffff0000u);
}

template <typename S>
__device__ __forceinline__ uint32_t narrow_word(const float *in);
template <>
__device__ __forceinline__ uint32_t narrow_word<float>(const float *in) {
  return __float_as_uint(in[0]);
}
template <>
__device__ __forceinline__ uint32_t narrow_word<__half>(const float *in) {
  return (uint32_t)__half_as_ushort(__float2half_rn(in[0])) |
         ((uint32_t)__half_as_ushort(__float2half_rn(in[1])) << 16);
}
template <>
__device__ __forceinline__ uint32_t narrow_word<bf16_t>(const float *in) {
  return float_to_bf16_bits(in[0]) | (float_to_bf16_bits(in[1]) << 16);
}

typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef double f64x2 __attribute__((ext_vector_type(2)));

// Two and four values of the arithmetic type as they lie in LDS.
template <typename R>
struct alignas(2 * sizeof(R)) Two {
  R x, y;
};
template <typename R>
struct alignas(16) Four {
  R x, y, z, w;
};

template <int BYTES>
struct Raw;
template <>
struct Raw<16> {
  using type = u32x4;
};
template <>
struct Raw<8> {
  using type = u32x2;
};
template <>
struct Raw<4> {
  using type = uint32_t;
};
template <>
struct Raw<2> {
  using type = uint16_t;
};

// Loads CNT elements of S (CNT*sizeof(S) in {2,4,8,16,32} bytes, 16-byte aligned from there on) in
// the arithmetic type.  STREAM marks data that is touched once (cost rows, upstream gradients):
// non-temporal.  GAP (double only): elements from one pair to the next, see lane_gap.
template <typename S, int CNT, bool STREAM, int GAP = 2>
__device__ __forceinline__ void load_vec(const S *p, typename Storage<S>::Real *out) {
  if constexpr (sizeof(S) == 8) {
    if constexpr (CNT == 1) {
      out[0] = STREAM ? __builtin_nontemporal_load(p) : *p;
    } else {
#pragma unroll
      for (int k = 0; k < CNT / 2; ++k) {
        const f64x2 *q = reinterpret_cast<const f64x2 *>(p + k * GAP);
        const f64x2 v = STREAM ? __builtin_nontemporal_load(q) : *q;
        out[2 * k] = v[0], out[2 * k + 1] = v[1];
      }
    }
  } else {
  constexpr int BYTES = CNT * (int)sizeof(S);
  using RawT = typename Raw<BYTES>::type;
  constexpr int PER_WORD = 4 / (int)sizeof(S);
  const RawT *q = reinterpret_cast<const RawT *>(p);
  const RawT v = STREAM ? __builtin_nontemporal_load(q) : *q;
  if constexpr (BYTES == 2) {
    float two[2];
    widen_word<S>(v, two);
    out[0] = two[0];
  } else if constexpr (BYTES == 4) {
    widen_word<S>(v, out);
  } else {
#pragma unroll
    for (int k = 0; k < BYTES / 4; ++k) widen_word<S>(v[k], out + k * PER_WORD);
  }
  }
}

// Output rows bypass the caches (non-temporal, STREAM) only where one store of a pixel's lanes covers
// whole 128-byte lines.  A narrower row -- 16 channels of a 16-bit type, a few correlation
// groups, the one mask word of a voxel -- shares its line with the rows of the neighbouring
// depths, which other store instructions write: streamed, each piece reaches memory on its own
// as a partial line, while L2 puts the pieces of a cached line together first (the
// valid-view counts of the MVSNet-stage forward: 134 -> 123 us).
template <typename S, int CNT, bool STREAM, int GAP = 2>
__device__ __forceinline__ void store_vec(S *p, const typename Storage<S>::Real *in) {
  if constexpr (sizeof(S) == 8) {
    if constexpr (CNT == 1) {
      if (STREAM) __builtin_nontemporal_store(in[0], p);
      else *p = in[0];
    } else {
#pragma unroll
      for (int k = 0; k < CNT / 2; ++k) {
        f64x2 *q = reinterpret_cast<f64x2 *>(p + k * GAP);
        const f64x2 v = {in[2 * k], in[2 * k + 1]};
        if (STREAM) __builtin_nontemporal_store(v, q);
        else *q = v;
      }
    }
  } else {
  constexpr int BYTES = CNT * (int)sizeof(S);
  using RawT = typename Raw<BYTES>::type;
  constexpr int PER_WORD = 4 / (int)sizeof(S);
  RawT *q = reinterpret_cast<RawT *>(p);
  RawT v;
  if constexpr (BYTES == 2) {
    float two[2] = {in[0], 0.f};
    v = (uint16_t)(narrow_word<S>(two) & 0xffffu);
  } else if constexpr (BYTES == 4) {
    v = narrow_word<S>(in);
  } else {
#pragma unroll
    for (int k = 0; k < BYTES / 4; ++k) v[k] = narrow_word<S>(in + k * PER_WORD);
  }
  if (STREAM)
    __builtin_nontemporal_store(v, q);
  else
    *q = v;
  }
}

// The same load without the conversion: CNT elements as they lie in memory, in 32-bit words
// (a single 16-bit element in the low half of one word).  A wave that widens 16-bit values
// right after the load waits for memory at that point; keeping the words and widening them
// where they are used lets the wait fall behind whatever work sits in between.
// (doubles are kept as doubles)
template <typename S>
using RawWord = typename std::conditional<sizeof(S) == 8, double, uint32_t>::type;
template <typename S, int CNT>
constexpr int raw_words() { return (CNT * (int)sizeof(S) + 3) / (int)sizeof(RawWord<S>); }
__device__ __forceinline__ float raw_to_real(uint32_t w) { return __uint_as_float(w); }
__device__ __forceinline__ double raw_to_real(double w) { return w; }
template <typename S, int CNT, bool STREAM, int GAP = 2>
__device__ __forceinline__ void load_raw(const S *p, RawWord<S> *out) {
  if constexpr (sizeof(S) == 8) {
    load_vec<S, CNT, STREAM, GAP>(p, out);
  } else {
  constexpr int BYTES = CNT * (int)sizeof(S);
  using RawT = typename Raw<BYTES>::type;
  const RawT *q = reinterpret_cast<const RawT *>(p);
  const RawT v = STREAM ? __builtin_nontemporal_load(q) : *q;
  if constexpr (BYTES <= 4) {
    out[0] = (uint32_t)v;
  } else {
#pragma unroll
    for (int k = 0; k < BYTES / 4; ++k) out[k] = v[k];
  }
  }
}
template <typename S, int CNT>
__device__ __forceinline__ void widen_raw(const RawWord<S> *in, typename Storage<S>::Real *out) {
  if constexpr (sizeof(S) == 8) {
#pragma unroll
    for (int k = 0; k < CNT; ++k) out[k] = in[k];
  } else {
  constexpr int BYTES = CNT * (int)sizeof(S);
  constexpr int PER_WORD = 4 / (int)sizeof(S);
  if constexpr (BYTES == 2) {
    float two[2];
    widen_word<S>(in[0], two);
    out[0] = two[0];
  } else {
#pragma unroll
    for (int k = 0; k < BYTES / 4; ++k) widen_word<S>(in[k], out + k * PER_WORD);
  }
  }
}

// (the choice is made at compile time from the row's width: a run-time test in front of every
// row store cost the MVSNet-stage forward 20 us)
constexpr bool whole_lines(int elements, int elem_bytes) { return elements * elem_bytes >= 128; }

// Which channels a lane owns.  Four consecutive ones, 16 bytes in float.  In double four would be 32
// bytes, which one access cannot move: each of two accesses of a pixel's lanes would touch every
// other 16 bytes of the row, and a streamed row would leave as half lines.  So in double a lane
// owns two pairs, one in each half of the row (channels 2 cl and half + 2 cl), and every access
// of a pixel is one contiguous run.  Not where a lane's channels have to be neighbours (correlation
// groups) and not with idle lanes (their pairs would lie in the other half).
constexpr int lane_gap(int lpp, int corr, int elem_bytes, bool pad) {
  return elem_bytes == 8 && corr != 1 && corr != 3 && corr != 5 && !pad ? 2 * lpp : 2;
}
// first channel of lane `cl`; channel c (0..3) is that + c / 2 * gap + c % 2
__device__ __forceinline__ int lane_first(int cl, int gap) { return gap == 2 ? cl * 4 : cl * 2; }

// This lane's four channels of an LDS row of channels (at `p`: the first).
template <int GAP, typename R>
__device__ __forceinline__ void slot_read(const R *p, R (&v)[4]) {
  if constexpr (sizeof(R) == 4) {
    const Four<R> w = *reinterpret_cast<const Four<R> *>(p);
    v[0] = w.x, v[1] = w.y, v[2] = w.z, v[3] = w.w;
  } else {
    const Two<R> lo = *reinterpret_cast<const Two<R> *>(p), hi = *reinterpret_cast<const Two<R> *>(p + GAP);
    v[0] = lo.x, v[1] = lo.y, v[2] = hi.x, v[3] = hi.y;
  }
}
template <int GAP, typename R>
__device__ __forceinline__ void slot_write(R *p, const R (&v)[4]) {
  if constexpr (sizeof(R) == 4) {
    *reinterpret_cast<Four<R> *>(p) = Four<R>{v[0], v[1], v[2], v[3]};
  } else {
    *reinterpret_cast<Two<R> *>(p) = Two<R>{v[0], v[1]};
    *reinterpret_cast<Two<R> *>(p + GAP) = Two<R>{v[2], v[3]};
  }
}

// An LDS object at (lane-dependent byte offset) + (compile-time constant).
template <typename T>
__device__ __forceinline__ T &lds_at(unsigned char *base, unsigned lane_bytes, int const_bytes) {
  return *reinterpret_cast<T *>(base + lane_bytes + const_bytes);
}

// Orders this wave's LDS traffic: the lanes of a wavefront execute in lockstep and the
// LDS returns a wave's operations in issue order, so only the compiler has to be kept
// from moving accesses across the phase boundary.
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Sum over each group of WIDTH consecutive lanes (WIDTH a power of two <= 16), left in every
// lane of the group.  Cross-lane moves in registers: quad permutes, then the half-row and
// row mirrors (a mirror pairs lane i with lane WIDTH-1-i; the quad steps finish the sum).
template <int CTRL>
__device__ __forceinline__ int dpp_move(int v) {
  return __builtin_amdgcn_mov_dpp(v, CTRL, 0xf, 0xf, true);
}
template <int CTRL>
__device__ __forceinline__ float dpp_move(float v) {
  return __int_as_float(dpp_move<CTRL>(__float_as_int(v)));
}
template <int CTRL>
__device__ __forceinline__ double dpp_move(double v) {
  return __hiloint2double(dpp_move<CTRL>(__double2hiint(v)), dpp_move<CTRL>(__double2loint(v)));
}
template <int CTRL, typename R>
__device__ __forceinline__ R dpp_add(R v) { return v + dpp_move<CTRL>(v); }
template <int WIDTH, typename R>
__device__ __forceinline__ R group_sum(R v) {
  static_assert(WIDTH == 1 || WIDTH == 2 || WIDTH == 4 || WIDTH == 8 || WIDTH == 16, "group width");
  if constexpr (WIDTH >= 16) v = dpp_add<0x140>(v);  // row_mirror
  if constexpr (WIDTH >= 8) v = dpp_add<0x141>(v);   // row_half_mirror
  if constexpr (WIDTH >= 4) v = dpp_add<0x4E>(v);    // quad_perm 2,3,0,1
  if constexpr (WIDTH >= 2) v = dpp_add<0xB1>(v);    // quad_perm 1,0,3,2
  return v;
}

// Sums the per-channel values of each correlation group: out[g] for g < VEC/sub.
template <int VEC, typename R>
__device__ __forceinline__ void fold_groups(const R *ch, int sub, R *out) {
  if (sub == 1) {
#pragma unroll
    for (int c = 0; c < VEC; ++c) out[c] = ch[c];
  } else if (sub == 2) {
#pragma unroll
    for (int c = 0; c < VEC / 2; ++c) out[c] = ch[2 * c] + ch[2 * c + 1];
  } else if (sub == 4) {
#pragma unroll
    for (int c = 0; c < VEC / 4; ++c)
      out[c] = (ch[4 * c] + ch[4 * c + 1]) + (ch[4 * c + 2] + ch[4 * c + 3]);
  } else {  // sub == 8: two lanes of four channels, both left with the sum
    static_assert(VEC == 4, "a group of eight is two lanes");
    out[0] = dpp_add<0xB1>((ch[0] + ch[1]) + (ch[2] + ch[3]));  // quad_perm 1,0,3,2
  }
}

// In double the rows of 16 channels, and those of groups of one channel, leave in two stores that touch half
// of every line each.  Streamed, the halves reach memory on their own as partial lines, which costs up to
// twice the time where little else goes on -- one or two views, or a row for every view: these ask the
// launcher (Geometry::stream_halves).  With more views the rows come seldom enough and streaming stays 5 to
// 10 % ahead of the caches.
constexpr bool half_lines(int lpp, int nv, int corr, int elem_bytes, bool pad) {
  return elem_bytes == 8 && !pad && lpp >= 4 &&
         ((corr == 1 && (nv == 1 || (nv == 2 && lpp >= 8))) || (lpp == 4 && (corr == 4 || (corr == 0 && nv == 1))));
}
template <typename S, int CNT, bool STREAM, bool ASK, int GAP = 2>
__device__ __forceinline__ void store_row(S *p, const typename Storage<S>::Real *v, bool stream) {
  if constexpr (ASK) {
    // (uniform; the two empty statements keep the compiler from making one store of the two, which
    // would be one that does not stream)
    if (stream) {
      asm volatile("");
      store_vec<S, CNT, true, GAP>(p, v);
      asm volatile("");
    } else {
      store_vec<S, CNT, false, GAP>(p, v);
    }
  } else {
    store_vec<S, CNT, STREAM, GAP>(p, v);
  }
}

template <typename S, int VEC, int LPP, bool PAD, bool ASK>
__device__ __forceinline__ void store_groups(S *p, const typename Storage<S>::Real *v, int sub, bool stream) {
  // p already points at this lane's first group; a pixel's row holds VEC * LPP / sub values
  constexpr int C = VEC * LPP, B = (int)sizeof(S);
  if (sub == 1) {
    store_row<S, VEC, !PAD && whole_lines(C, B), ASK>(p, v, stream);
  } else if (sub == 2) {
    store_vec<S, VEC / 2, !PAD && whole_lines(C / 2, B)>(p, v);
  } else if (sub == 4) {
    store_vec<S, VEC / 4, !PAD && whole_lines(C / 4, B)>(p, v);
  } else if (threadIdx.x & 1) {  // sub == 8: the group's second lane
    store_vec<S, 1, !PAD && whole_lines(C / 8, B)>(p, v);
  }
}

// Offset of lane `cl`'s first group in a row of group values (a group of eight: lanes 2g, 2g + 1).
template <int VEC>
__device__ __forceinline__ int group_offset(int cl, int sub) {
  return sub == 8 ? cl >> 1 : cl * (VEC / sub);
}

// ---- shared front end of both kernels ---------------------------------------------------
template <int NV, typename R>
struct Cameras {
  R zc[NV], wc[NV], hc[NV];  // rows of R applied to (ref_w, ref_h, 1)
  R t0[NV], t1[NV], t2[NV];
};

template <int LPP>
struct Tile {
  int lane, p, cl;
  int b, pin, h, w;
  int d_lo, d_hi;
  int view0;               // first view of this workgroup's group
  bool pix_ok;
  int64_t pix;
};

template <typename S, int LPP, bool TALL = false>
__device__ __forceinline__ bool locate_tile(const Args<S> &a, const Geometry &g, Tile<LPP> &t) {
  constexpr int PPW = 64 / LPP;
  t.lane = threadIdx.x;
  // Workgroups are dealt round-robin to the 8 XCDs; give each XCD runs of consecutive
  // tiles so that its L2 only has to hold that part of the source images.  Forward: one
  // band per XCD.  Backward: short runs, which balance the XCDs better (its tiles differ
  // more in cost).
  // (all counts fit 32 bits: the host checks total_units; 64-bit divisions would cost
  // several hundred instructions per workgroup, which runs only a few thousand)
  const unsigned bid = blockIdx.x;
  const unsigned r = bid >> 3, x = bid & 7u;
  const unsigned unit = g.xcd_shift < 0
                            ? x * (unsigned)g.units_per_xcd + r
                            : ((r >> g.xcd_shift) << (g.xcd_shift + 3)) + (x << g.xcd_shift) +
                                  (r & ((1u << g.xcd_shift) - 1u));
  // (pixels of one and two lanes never come segment by segment, see make_geometry)
  const bool by_segment = LPP >= 4 && g.xcd_shift == kBandsBySegment;
  if (!by_segment && unit >= (unsigned)g.total_units) return false;
  // the groups of one (tile, segment) are neighbours in launch order: they stream the same
  // upstream-gradient rows at about the same time, through the same L2
  unsigned tile;
  int segi;
  if (g.xcd_shift >= 0) {
    // Backward: the depth segments one after the other, all tiles of the first segment first.
    // The workgroups of a launch differ in length, and what the chip does while the last ones
    // finish is lost; the segment of the nearest hypotheses (most cell changes per depth) is
    // the longest, so it goes first and the launch ends on the shortest workgroups
    // (MVSNet-stage backward -2.5 %; the far segment first: +0.5 %).
    const unsigned sraw = unit / g.units_per_seg;
    const unsigned rem = unit - sraw * g.units_per_seg;
    segi = (int)sraw;
    tile = rem / (unsigned)g.ngroups;
    t.view0 = (int)(rem - tile * (unsigned)g.ngroups) * g.vper;
  } else {
    // (one view group.  One division for both orders: a unit into tile and segment, or a place in an
    // XCD's launches into segment and tile of its band)
    const unsigned num = by_segment ? r : unit, den = by_segment ? (unsigned)g.units_per_xcd : (unsigned)g.nseg;
    const unsigned quot = num / den, rem = num - quot * den;
    tile = by_segment ? x * den + rem : quot;
    segi = (int)(by_segment ? quot : rem);
    t.view0 = 0;
    if (by_segment && tile >= g.units_per_seg) return false;
  }
  t.d_lo = segi * g.seg;
  t.d_hi = min((int)a.D, t.d_lo + g.seg);
  t.b = (int)(tile / (unsigned)g.tiles_per_image);
  const int t_in = (int)(tile - (unsigned)t.b * (unsigned)g.tiles_per_image);
  t.p = t.lane / LPP;
  t.cl = t.lane % LPP;
  if constexpr (PPW == 1) {
    t.pin = t_in;
    t.pix_ok = true;
  } else {
    // A tile is tile_rows(PPW) rows of pixels: the samples of a compact tile cross texel boundaries
    // at more nearly the same depths than those of a long row, so fewer wave iterations carry
    // a cell change (0.49 against 0.62 of them on the MVSNet-stage workload).  Tiles that
    // stick out of the image have their outside pixels switched off.
    constexpr int TH = tile_rows(PPW, TALL), TW = PPW / TH;
    const int ty = t_in / g.tiles_x, tx = t_in - ty * g.tiles_x;
    const int py = t.p / TW;
    const int y = ty * TH + py, x = tx * TW + (t.p - py * TW);
    t.pix_ok = y < (int)a.H && x < (int)a.W;
    t.pin = y * (int)a.W + x;
  }
  if (!t.pix_ok) t.pin = g.hw - 1;  // clamp: loads stay in range, stores are predicated
  t.pix = (int64_t)t.b * g.hw + t.pin;
  t.h = t.pin / (int)a.W;
  t.w = t.pin - t.h * (int)a.W;
  return true;
}

template <typename S, int NV>
__device__ __forceinline__ void load_cameras(const Args<S> &a, int b, int view0,
                                             typename Storage<S>::Real ref_w,
                                             typename Storage<S>::Real ref_h,
                                             Cameras<NV, typename Storage<S>::Real> &c) {
  const int N = (int)a.N;
#pragma unroll
  for (int n = 0; n < NV; ++n) {
    const int nn = view0 + n < N ? view0 + n : 0;
    const auto *Rm = a.Rs + ((int64_t)b * N + nn) * 9;
    const auto *t = a.Ts + ((int64_t)b * N + nn) * 3;
    // same association as the per-voxel expression: (R6*w + R7*h) + R8
    c.zc[n] = Rm[6] * ref_w + Rm[7] * ref_h + Rm[8];
    c.wc[n] = Rm[0] * ref_w + Rm[1] * ref_h + Rm[2];
    c.hc[n] = Rm[3] * ref_w + Rm[4] * ref_h + Rm[5];
    c.t0[n] = t[0], c.t1[n] = t[1], c.t2[n] = t[2];
  }
}

// w / z and h / z, each correctly rounded, with one reciprocal between them.  The steps are those of a
// correctly rounded division by Newton's iteration and residual corrections (Markstein, "Computation of
// elementary functions on the IBM RISC System/6000 processor", 1990), without the scaling that only divisors
// and quotients at the ends of the exponent's range need: fourteen operations (double: twelve) where two
// divisions are twenty-two.  Divisors outside 2^-60 .. 2^60 (double: 2^-500 .. 2^500) make the wave divide
// the plain way, and `small`: quotients near zero matter too (without it one below a quarter, which no
// caller accepts, may be off).
__device__ __forceinline__ bool unusual_divisor(float z) { return __float_as_uint(z) - 0x21800000u > 0x3c000000u; }
__device__ __forceinline__ bool unusual_divisor(double z) { return (unsigned)__double2hiint(z) - 0x20b00000u > 0x3e800000u; }
__device__ __forceinline__ void quotients(float w, float h, float z, bool small, float &qw, float &qh) {
  float r = __builtin_amdgcn_rcpf(z);
  r = __builtin_fmaf(__builtin_fmaf(-z, r, 1.f), r, r);
  qw = w * r, qh = h * r;
  qw = __builtin_fmaf(__builtin_fmaf(-z, qw, w), r, qw);
  qh = __builtin_fmaf(__builtin_fmaf(-z, qh, h), r, qh);
  qw = __builtin_fmaf(__builtin_fmaf(-z, qw, w), r, qw);
  qh = __builtin_fmaf(__builtin_fmaf(-z, qh, h), r, qh);
  if (small || __ballot(unusual_divisor(z)) != 0ull) qw = w / z, qh = h / z;
}
__device__ __forceinline__ void quotients(double w, double h, double z, bool small, double &qw, double &qh) {
  double r = __builtin_amdgcn_rcp(z);
  r = __builtin_fma(__builtin_fma(-z, r, 1.0), r, r);
  r = __builtin_fma(__builtin_fma(-z, r, 1.0), r, r);
  qw = w * r, qh = h * r;
  qw = __builtin_fma(__builtin_fma(-z, qw, w), r, qw);
  qh = __builtin_fma(__builtin_fma(-z, qh, h), r, qh);
  if (small || __ballot(unusual_divisor(z)) != 0ull) qw = w / z, qh = h / z;
}
__device__ __forceinline__ float fraction(float x) { return __builtin_amdgcn_fractf(x); }  // x - floor(x), exact for x >= 0
__device__ __forceinline__ double fraction(double x) { return __builtin_amdgcn_fract(x); }

// One reprojection with hoisted row products; bit-identical to warp.h's project().
template <typename R>
struct Hit {
  int cell;    // place of tap (fh,fw) in the view's image, or -1: not accepted, the rest means nothing
  int key;     // (fh << 16) | fw
  R k00, k01, k11, k10;
  R dh, dw;
  R z, w3d, h3d;
};

// Without branches: what a rejected sample leaves behind is never looked at.  `wanted`: this lane's voxel counts.
// (image rows and columns fit 15 bits, see make_plan.)  With the shared reciprocal, 24-bit products, taps
// addressed from a uniform base and the window's four slot numbers put together by byte permutes a view of a
// chunk takes about 60 instructions less than it did (of 170 in the gradients, of 74 forward), and the forward
// kernels up to nine registers: gradients -2 to -8 % (f16, 16 channels, four views, 256 x 320 x 32, 235 -> 219
// us; 16-channel minimum, three views, 259 -> 244), forward 0 to -15 % (bf16 groups, four views, 512 x 640 x
// 8, 137 -> 129 us; CostAggregate's minimum of 16 channels, four views, 69 -> 60).
template <int NV, typename R>
__device__ __forceinline__ void reproject(const Cameras<NV, R> &c, int n, R depth, R half, R src_h_max, R src_w_max,
                                          int srcW, bool wanted, Hit<R> &r) {
  r.z = c.zc[n] * depth + c.t2[n];
  r.w3d = c.wc[n] * depth + c.t0[n];
  r.h3d = c.hc[n] * depth + c.t1[n];
  R sw, sh;
  quotients(r.w3d, r.h3d, r.z, half == R(0), sw, sh);
  sw = sw - half;
  sh = sh - half;
  const bool ok = wanted && !(r.z <= R(0)) && sh > R(0) && sw > R(0) && sh < src_h_max && sw < src_w_max;
  const int fh = static_cast<int>(sh), fw = static_cast<int>(sw);
  r.dh = fraction(sh);
  r.dw = fraction(sw);
  const R eh = R(1) - r.dh, ew = R(1) - r.dw;
  r.k11 = r.dh * r.dw;
  r.k10 = r.dh * ew;
  r.k00 = eh * ew;
  r.k01 = eh * r.dw;
  r.cell = ok ? (int)__umul24((unsigned)fh, (unsigned)srcW) + fw : -1;
  r.key = (fh << 16) | (fw & 0xffff);
}

// Four taps of a cell, this lane's channels, in the arithmetic type -- or (RAW, f16 under a mean) as loaded: a
// multiply-add takes half-precision factors as they are (v_fma_mix_f32, the same single rounding), so the
// sixteen conversions at every cell change, which wait for the loads, and half the registers are not needed.
// (f16: cascade stage, four views of 16 channels, 256 x 320 x 32, gradient 219 -> 201 us, forward 85 -> 78; 32
// channels, two views, 128 x 160 x 96, 172 -> 164 and 61 -> 57; 8 channels, four views, 512 x 640 x 8, 67 -> 60.)
// Literal forms round the product by itself, which costs them a conversion per depth: they keep the widened taps.
template <typename S, int VEC, bool RAW = false>
struct Taps {
  typename Storage<S>::Real v[4][VEC];
  __device__ __forceinline__ typename Storage<S>::Real operator()(int k, int c) const { return v[k][c]; }
  template <int GAP>
  __device__ __forceinline__ void load(int k, const S *p) { load_vec<S, VEC, false, GAP>(p, v[k]); }
};
template <int VEC>
struct Taps<__half, VEC, true> {
  uint32_t w[4][VEC / 2];
  __device__ __forceinline__ float operator()(int k, int c) const {
    return __half2float(__ushort_as_half((unsigned short)(c & 1 ? w[k][c / 2] >> 16 : w[k][c / 2] & 0xffffu)));
  }
  template <int GAP>
  __device__ __forceinline__ void load(int k, const __half *p) { load_raw<__half, VEC, false, GAP>(p, w[k]); }
};
template <typename S>
constexpr bool is_half() { return std::is_same<S, __half>::value; }

// The four taps (00, 01, 11, 10) of a cell, this lane's channels: the view's uniform base and 32 bits of
// bytes (an image has less than 2^29 elements, make_plan).  `cell` counts units of UNIT elements: texels, or
// elements where the channel count is a run-time value (its product is then formed once per voxel).
constexpr int cell_unit(int channels, bool pad) { return pad ? 1 : channels; }
template <typename S, int VEC, int GAP, int UNIT, bool RAW>
__device__ __forceinline__ void load_cell(const S *view, int cell, int C, int row_step, unsigned lane_ch,
                                          Taps<S, VEC, RAW> &tap) {
  const unsigned e0 = ((unsigned)cell * (unsigned)UNIT + lane_ch) * (unsigned)sizeof(S);
  const unsigned e1 = e0 + (unsigned)row_step * (unsigned)sizeof(S);
  const char *base = reinterpret_cast<const char *>(view);
  const unsigned step = (unsigned)C * (unsigned)sizeof(S);
  // (the texel to the right at a distance known when compiling lands in the instruction's offset field)
  const char *row0 = base + e0, *row1 = base + e1;
  const char *right0 = UNIT > 1 ? row0 + UNIT * sizeof(S) : base + (e0 + step);
  const char *right1 = UNIT > 1 ? row1 + UNIT * sizeof(S) : base + (e1 + step);
  tap.template load<GAP>(0, reinterpret_cast<const S *>(row0));
  tap.template load<GAP>(1, reinterpret_cast<const S *>(right0));
  tap.template load<GAP>(2, reinterpret_cast<const S *>(right1));
  tap.template load<GAP>(3, reinterpret_cast<const S *>(row1));
}

template <typename S>
__device__ __forceinline__ typename Storage<S>::Real voxel_depth(const Args<S> &a, int64_t pix, int b,
                                                                 int d,
                                                                 typename Storage<S>::Real base) {
  return a.depth_grid ? a.depth_grid[pix * a.D + d] : base + a.offsets[(int64_t)b * a.D + d];
}

// =========================================================================================
// Forward
// =========================================================================================
// Stores CNT (1, 2 or 4) consecutive int32 values; STREAM as for the cost rows.
template <int CNT, bool STREAM>
__device__ __forceinline__ void store_ints(int32_t *p, const int *v) {
  constexpr bool stream = STREAM;
  if constexpr (CNT == 4) {
    typedef int i32x4 __attribute__((ext_vector_type(4)));
    i32x4 w = {v[0], v[1], v[2], v[3]};
    if (stream) __builtin_nontemporal_store(w, reinterpret_cast<i32x4 *>(p));
    else *reinterpret_cast<i32x4 *>(p) = w;
  } else if constexpr (CNT == 2) {
    typedef int i32x2 __attribute__((ext_vector_type(2)));
    i32x2 w = {v[0], v[1]};
    if (stream) __builtin_nontemporal_store(w, reinterpret_cast<i32x2 *>(p));
    else *reinterpret_cast<i32x2 *>(p) = w;
  } else {
    if (stream) __builtin_nontemporal_store(v[0], p);
    else *p = v[0];
  }
}

// A row of winners per channel, four of this lane's.
template <int VEC, int LPP, int GAP, bool PAD>
__device__ __forceinline__ void store_winners(int32_t *p, const int *v) {
  if constexpr (GAP == 2) {
    store_ints<VEC, !PAD && whole_lines(VEC * LPP, 4)>(p, v);
  } else {
    store_ints<2, false>(p, v);
    store_ints<2, false>(p + GAP, v + 2);
  }
}

// ---- CostVolumeV3: the largest correlation of any source group with any reference group ------
// The mean over k accepted views.  In its literal form the division rounds like the reference's:
// halving and quartering are exact, so only other counts pay for one.
template <bool LIT, typename R>
__device__ __forceinline__ void mean_of(R (&acc)[4], int k) {
  if constexpr (LIT) {
    if (k == 2 || k == 4) {
      const R part = k == 2 ? R(0.5) : R(0.25);
#pragma unroll
      for (int c = 0; c < 4; ++c) acc[c] *= part;
    } else if (k > 2) {
#pragma unroll
      for (int c = 0; c < 4; ++c) acc[c] /= static_cast<R>(k);
    }
  } else if (k > 1) {
    const R inv = quick_recip(static_cast<R>(k));
#pragma unroll
    for (int c = 0; c < 4; ++c) acc[c] *= inv;
  }
}
// The group values of a lane: its channels' sums folded, or (literal form, add_groups) already so.
template <bool LIT, typename R>
__device__ __forceinline__ void fold_or_keep(const R (&acc)[4], int sub, R (&out)[4]) {
  if constexpr (LIT) {
#pragma unroll
    for (int c = 0; c < 4; ++c) out[c] = acc[c];
  } else {
    fold_groups<4>(acc, sub, out);
  }
}
// One butterfly step of "largest value, earliest pair on a tie" (both partners end equal).
template <int CTRL, typename R>
__device__ __forceinline__ void better_pair(R &best, int &code) {
  const R ob = dpp_move<CTRL>(best);
  const int oc = dpp_move<CTRL>(code);
  const bool take = ob > best || (ob == best && oc < code);
  best = take ? ob : best;
  code = take ? oc : code;
}
// A group of eight channels held by two lanes: the odd lane continues the even lane's sum over
// its own four, in channel order (the result of the odd lane is the group's).
template <typename R>
__device__ __forceinline__ R continue_group(R sum, const R (&val)[4], int cl) {
  const R head = dpp_move<0xA0>(sum);  // quad_perm 0,0,2,2
  return (cl & 1) ? (((head + val[0]) + val[1]) + val[2]) + val[3] : sum;
}
// The maximum reduce of one accepted view: where a correlation group of this lane is larger than
// the largest so far (strictly: the earliest view keeps a tie), it and its view are kept.  A
// group's products are summed in channel order.  One branch on the group width per sample (the
// width is a run-time value; picking the terms of every group by comparisons instead took, with
// the wave per SIMD of forward_min_waves, 157 against 140 us on an f16 sweep of 32 channels in
// eight groups, four views, 237 x 315 x 24).
template <typename R>
__device__ __forceinline__ void keep_larger_groups(R (&best)[4], int (&arg)[4], const R (&val)[4],
                                                   int sub, int cl, int view) {
  auto keep = [&](int i, R corr) __attribute__((always_inline)) {
    if (best[i] < corr) best[i] = corr, arg[i] = view;
  };
  if (sub >= 4) {
    R corr = ((val[0] + val[1]) + val[2]) + val[3];
    if (sub == 8) corr = continue_group(corr, val, cl);
    keep(0, corr);
  } else if (sub == 2) {
    keep(0, val[0] + val[1]);
    keep(1, val[2] + val[3]);
  } else {
#pragma unroll
    for (int c = 0; c < 4; ++c) keep(c, val[c]);
  }
}
// The mean's literal form: one view's products, added up group by group in channel order, join the
// sums of the views before it.
template <typename R>
__device__ __forceinline__ void add_groups(R (&acc)[4], const R (&val)[4], int sub, int cl) {
  if (sub >= 4) {
    R corr = ((val[0] + val[1]) + val[2]) + val[3];
    if (sub == 8) corr = continue_group(corr, val, cl);
    acc[0] += corr;
  } else if (sub == 2) {
    acc[0] += val[0] + val[1];
    acc[1] += val[2] + val[3];
  } else {
#pragma unroll
    for (int c = 0; c < 4; ++c) acc[c] += val[c];
  }
}
constexpr int kNoPair = 0x7fffffff;
constexpr int kPairRow = 64;  // pair code: source group * kPairRow + reference group
// Largest value and smallest integer over the lanes of a pixel, left in every one of them (a NaN
// gives way to a number: one instruction each, the lane move is part of it).
__device__ __forceinline__ float larger(float a, float b) { return __builtin_fmaxf(a, b); }
__device__ __forceinline__ double larger(double a, double b) { return __builtin_fmax(a, b); }
template <int LPP, typename R>
__device__ __forceinline__ R group_max(R v) {
  if constexpr (LPP >= 2) v = larger(v, dpp_move<0xB1>(v));
  if constexpr (LPP >= 4) v = larger(v, dpp_move<0x4E>(v));
  if constexpr (LPP >= 8) v = larger(v, dpp_move<0x141>(v));
  if constexpr (LPP >= 16) v = larger(v, dpp_move<0x140>(v));
  return v;
}
template <int LPP>
__device__ __forceinline__ int group_min(int v) {
  if constexpr (LPP >= 2) v = min(v, dpp_move<0xB1>(v));
  if constexpr (LPP >= 4) v = min(v, dpp_move<0x4E>(v));
  if constexpr (LPP >= 8) v = min(v, dpp_move<0x141>(v));
  if constexpr (LPP >= 16) v = min(v, dpp_move<0x140>(v));
  return v;
}
// (CORR 3: groups of four and eight channels; CORR 5: of one and two)
constexpr bool best_pair_op(int corr) { return corr == 3 || corr == 5; }

// The best (source group, reference group) pair of one accepted sample of one pixel, found
// by the pixel's LPP lanes exactly as the reference's loop finds it
// (cost_volume_kernels_gpu_v3.cu.cc:113-130): lane cl holds the sample of channels
// 4cl..4cl+3, i.e. part (cl % (SUB/4)) of group cl / (SUB/4); every dot product is one
// sequential chain over the group's channels, each product and sum rounded separately (for 8
// channels the even lane's partial sum continues in the odd lane); source group outermost,
// strict "<" from the smallest positive float, so the earliest pair keeps a tie.
// `ref_row`: the pixel's reference channels in LDS.  Every lane of the pixel returns the same
// best value (the seed when no pair exceeds it) and pair code (kNoPair then).
// Every pair is one thread's own loop in the general kernel, which these widths and double ran before
// (groups of one, two views, 41 x 54 x 9, two images of 32 channels: forward 360 -> 11 us, gradient 380
// -> 32 us; double, groups of two, three views, 213 x 309 x 33: 2330 -> 1045 and 3700 -> 1570 us).  One
// class loses: the minimum's gradient of narrow groups over a large image and two views (383 x 534 x
// 27: 1090 -> 1250 us, with a forward pass of 6100 -> 300 us), where few channels receive anything.
// Groups of two channels: a lane's four are two source groups.  Groups of one (every channel with every
// channel): the largest product of a source value is with the pixel's largest reference value, or with
// its smallest where the source value is negative, because rounding keeps the order; so `ends` (the
// two, ref_ends) replace the search, and the pair is then the first source channel and the first
// reference channel whose product is that value.
template <typename R, int VEC, int LPP, int SUB, bool CODE>
__device__ __forceinline__ void v3_best_pair(const R (&smp)[VEC], const R *ref_row, const Two<R> &ends, int cl,
                                             R &best, int &code) {
  static_assert(VEC == 4 && (SUB == 1 || SUB == 2 || SUB == 4 || SUB == 8), "a group: part of a lane, one lane or two");
  constexpr int C = VEC * LPP, G = C / SUB, LPG = SUB <= 4 ? 1 : SUB / 4;
  const int group = SUB >= 4 ? cl / LPG : cl * (4 / SUB), koff = (cl % LPG) * 4;
  best = Limits<R>::min_positive();
  code = kNoPair;
  if constexpr (SUB == 1) {
    R top[VEC];
#pragma unroll
    for (int c = 0; c < VEC; ++c) {
      top[c] = smp[c] * (smp[c] > R(0) ? ends.y : ends.x);
      best = larger(best, top[c]);
    }
    best = group_max<LPP>(best);
    if constexpr (!CODE) return;
    int gs = kNoPair;
#pragma unroll
    for (int c = VEC - 1; c >= 0; --c)
      if (top[c] == best) gs = group + c;
    gs = group_min<LPP>(gs);
    if (gs != kNoPair) {  // (the seed itself may equal a product: such a pair does not exceed it)
      const int cs = gs & 3;
      const R own = cs == 0 ? smp[0] : cs == 1 ? smp[1] : cs == 2 ? smp[2] : smp[3];
      const R s = __shfl(own, gs >> 2, LPP);
      const Four<R> r = *reinterpret_cast<const Four<R> *>(ref_row + cl * 4);
      int gi = kNoPair;
      if (s * r.w == best) gi = group + 3;
      if (s * r.z == best) gi = group + 2;
      if (s * r.y == best) gi = group + 1;
      if (s * r.x == best) gi = group;
      gi = group_min<LPP>(gi);
      if (Limits<R>::min_positive() < best) code = gs * kPairRow + gi;
    }
    return;
  } else if constexpr (SUB == 2) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
#pragma unroll 4
      for (int g2 = 0; g2 < G; g2 += 2) {
        const Four<R> r = *reinterpret_cast<const Four<R> *>(ref_row + g2 * 2);
        const R d0 = smp[2 * u] * r.x + smp[2 * u + 1] * r.y, d1 = smp[2 * u] * r.z + smp[2 * u + 1] * r.w;
        if constexpr (CODE) {
          if (best < d0) best = d0, code = (group + u) * kPairRow + g2;
          if (best < d1) best = d1, code = (group + u) * kPairRow + g2 + 1;
        } else {
          best = larger(best, larger(d0, d1));
        }
      }
    }
    if constexpr (CODE) {
      if constexpr (LPP >= 2) better_pair<0xB1>(best, code);    // quad_perm 1,0,3,2
      if constexpr (LPP >= 4) better_pair<0x4E>(best, code);    // quad_perm 2,3,0,1
      if constexpr (LPP >= 8) better_pair<0x141>(best, code);   // row_half_mirror
      if constexpr (LPP >= 16) better_pair<0x140>(best, code);  // row_mirror
    } else {
      best = group_max<LPP>(best);
    }
  } else {
    // The largest value first (one instruction per pair, the lanes' tournament included), then the
    // first pair that has it: keeping value and pair together takes three and a longer tournament
    // (32 channels in four groups, two views, 120 x 152 x 64: forward, which needs no pair, 78 -> 60 us,
    // gradient 199 -> 189 us).
    R dot[G];
#pragma unroll
    for (int gi = 0; gi < G; ++gi) {
      const Four<R> r = *reinterpret_cast<const Four<R> *>(ref_row + gi * SUB + koff);
      const R p0 = smp[0] * r.x, p1 = smp[1] * r.y, p2 = smp[2] * r.z, p3 = smp[3] * r.w;
      dot[gi] = ((p0 + p1) + p2) + p3;  // (0 + p0 differs from p0 in the sign of zero only)
      if constexpr (LPG == 2) {
        const R head = dpp_move<0xA0>(dot[gi]);  // quad_perm 0,0,2,2: the even lane's four terms
        dot[gi] = (((head + p0) + p1) + p2) + p3;    // complete in the odd lane
      }
    }
    const bool mine = LPG == 1 || (cl & 1) != 0;
    R top = dot[0];
#pragma unroll
    for (int gi = 1; gi < G; ++gi) top = larger(top, dot[gi]);
    best = group_max<LPP>(larger(best, mine ? top : best));
    if constexpr (CODE) {
#pragma unroll
      for (int gi = G - 1; gi >= 0; --gi)
        if (dot[gi] == best) code = group * kPairRow + gi;
      code = group_min<LPP>(mine ? code : kNoPair);
      if (!(Limits<R>::min_positive() < best)) code = kNoPair;  // no pair exceeds the seed
    }
  }
}

// Smallest and largest reference value of a pixel, NaN apart.
template <int LPP, typename R>
__device__ __forceinline__ Two<R> ref_ends(const R (&ref)[4]) {
  const R hi = larger(larger(ref[0], ref[1]), larger(ref[2], ref[3]));
  const R lo = -larger(larger(-ref[0], -ref[1]), larger(-ref[2], -ref[3]));
  return Two<R>{-group_max<LPP>(-lo), group_max<LPP>(hi)};
}

// The gradient of one accepted sample flows through one pair: the view's best pair, found
// again as in the forward (REDUCE 0, :469-491), or the recorded winner `pair` (REDUCE 1).
// Out: gsrc = d(loss)/d(sample) of this lane's channels (zero outside the winning source
// group); racc += the reference gradient of this lane's channels (zero outside the winning
// reference group, :494-512).  `rows` = two LDS arrays of 64*VEC floats: the pixel rows of
// the reference image (written once by the caller) and of this sample.
template <typename R, int VEC, int LPP, int SUB, int REDUCE>
__device__ __forceinline__ void v3_pair_gradients(const Four<R> wt, const R (&tap)[4][VEC], const Two<R> &ends,
                                                  R cg, int pair, R *rows, int p, int cl,
                                                  R (&racc)[VEC], R (&gsrc)[VEC]) {
  constexpr int C = VEC * LPP, LPG = SUB <= 4 ? 1 : SUB / 4;
  R *ref_row = rows + p * C, *smp_row = rows + 64 * VEC + p * C;
  const int group = SUB >= 4 ? cl / LPG : cl * (4 / SUB), koff = (cl % LPG) * 4;
  R smp[VEC];
#pragma unroll
  for (int c = 0; c < 4; ++c)
    smp[c] = wt.x * tap[0][c] + wt.y * tap[1][c] + wt.z * tap[2][c] + wt.w * tap[3][c];
  *reinterpret_cast<Four<R> *>(smp_row + cl * 4) = Four<R>{smp[0], smp[1], smp[2], smp[3]};
  int code = pair;
  if constexpr (REDUCE == 0) {
    R best;
    v3_best_pair<R, VEC, LPP, SUB, true>(smp, ref_row, ends, cl, best, code);
  }
  const bool any = code != kNoPair;
  const int gi_w = any ? code % kPairRow : 0, gs_w = any ? code / kPairRow : 0;
#pragma unroll
  for (int c = 0; c < 4; ++c) gsrc[c] = R(0);
  if constexpr (SUB >= 4) {
    if (any && group == gs_w) {
      const Four<R> r = *reinterpret_cast<const Four<R> *>(ref_row + gi_w * SUB + koff);
      gsrc[0] = cg * r.x, gsrc[1] = cg * r.y, gsrc[2] = cg * r.z, gsrc[3] = cg * r.w;
    }
  } else {
#pragma unroll
    for (int c = 0; c < 4; ++c)
      if (any && group + c / SUB == gs_w) gsrc[c] = cg * ref_row[gi_w * SUB + c % SUB];
  }
  wave_sync();  // the sample row is complete
  if constexpr (SUB >= 4) {
    if (any && group == gi_w) {
      const Four<R> m = *reinterpret_cast<const Four<R> *>(smp_row + gs_w * SUB + koff);
      racc[0] = mad(cg, m.x, racc[0]), racc[1] = mad(cg, m.y, racc[1]);
      racc[2] = mad(cg, m.z, racc[2]), racc[3] = mad(cg, m.w, racc[3]);
    }
  } else {
#pragma unroll
    for (int c = 0; c < 4; ++c)
      if (any && group + c / SUB == gi_w) racc[c] = mad(cg, smp_row[gs_w * SUB + c % SUB], racc[c]);
  }
}

// The first workgroups of a forward launch read one word of every 128-byte line of the source
// and reference images, 128 lines per workgroup, so that the images stream into the memory-side
// cache at the start of the launch.  Without it a launch that finds them in no cache spends its
// first tens of microseconds on tap gathers that each wait for HBM (MVSNet-stage forward after
// the caches have been overwritten: 152 -> 127 us; no difference when the images are cached).
// Only for images of up to 16 MB together: larger ones do not stay in the caches anyway, and
// touching them costs the launch their size in extra reads (f16 cascade workload, 29 MB:
// forward 95 -> 107 us with it).
// The values are not used; keep_alive() at the end of the kernel keeps the loads in the code.
struct Touched {
  unsigned a, b;
};
template <typename S>
__device__ __forceinline__ Touched touch_images(const Args<S> &a) {
  Touched w{0u, 0u};
  const size_t src_bytes = (size_t)a.B * a.N * a.srcH * a.srcW * a.C * sizeof(S);
  const size_t ref_bytes = a.ref != nullptr ? (size_t)a.B * a.H * a.W * a.C * sizeof(S) : 0;
  const size_t o0 = ((size_t)blockIdx.x * 128 + threadIdx.x) * 128, o1 = o0 + 64 * 128;
  if (src_bytes + ref_bytes <= ((size_t)16 << 20) && o0 < src_bytes + ref_bytes) {  // (uniform)
    const char *sb = reinterpret_cast<const char *>(a.src), *rb = reinterpret_cast<const char *>(a.ref);
    if (o0 + 4 <= src_bytes)
      w.a = *reinterpret_cast<const unsigned *>(sb + o0);
    else if (o0 >= src_bytes && o0 - src_bytes + 4 <= ref_bytes)
      w.a = *reinterpret_cast<const unsigned *>(rb + (o0 - src_bytes));
    if (o1 + 4 <= src_bytes)
      w.b = *reinterpret_cast<const unsigned *>(sb + o1);
    else if (o1 >= src_bytes && o1 - src_bytes + 4 <= ref_bytes)
      w.b = *reinterpret_cast<const unsigned *>(rb + (o1 - src_bytes));
  }
  return w;
}
__device__ __forceinline__ void keep_alive(const Touched &w) {
  asm volatile("" ::"v"(w.a), "v"(w.b));  // no instruction: the two registers count as read here
}

template <int NV, typename R = float>
constexpr int forward_lds_bytes(int lpp) {
  return lpp > 1 ? NV * 64 * (4 * (int)sizeof(R) + 4) : 0;
}
// The sums of squares that have to be added up in channel order (the minimum, and the mean in its
// literal form) also stage one chunk of squares per view: a row of C (+4 padding, so that the
// readers of a pixel hit different banks) values per (pixel, depth).  From eight lanes on half the
// chunk's depths at a time: whole chunks are 9 KB (32 channels), in double 18 KB, which with the
// records held a CU to twelve workgroups and to five (minimum over three views, 135 x 181 x 48, 83 ->
// 67 us with the segments of choose_segments; double, mean over three views, 149 x 220 x 116, 607 ->
// 480 us).  Not with five and six views in float, whose registers hold the kernel to three waves
// anyway (five views, 108 x 126 x 77: 147 us, 157 in halves).
constexpr int squares_depths(int lpp, int nv, bool wide_real) {
  return lpp >= 8 && (wide_real || nv <= 4) ? lpp / 2 : lpp;
}
template <int NV, typename R = float>
constexpr int forward_squares_bytes(int lpp) {
  return lpp > 1 ? 64 / lpp * squares_depths(lpp, NV, sizeof(R) == 8) * (4 * lpp + 4) * (int)sizeof(R) : 0;
}

// REDUCE: 0 mean over the accepted views (mask = their number), 1 per-channel minimum of
// the squared difference / per-group maximum of the correlation with the winning view as
// mask (-1: none).  The winner must be the reference's, so that reduce uses the literal
// operand order with every operation rounded separately instead of the fused chains.
// Minimum waves per SIMD the register allocator has to leave room for (the mean, and the minimum /
// maximum of four views; elsewhere the winner indices per depth and channel would spill).  Five and six views: left alone the compiler takes ~140
// registers (three waves); held to 128 it needs no scratch, and the fourth wave hides the tap
// gathers of wide-baseline views (stress workload forward 5.17 -> 4.45 ms).  Three and four
// views at four lanes per pixel: 102 -> 87 registers without scratch, five waves instead of
// four (f16 cascade workload forward 122 -> 113 us cold); the other widths would spill.
// MIN / MAX of four views: 129-131 registers left alone, 8 bytes of scratch at 128 and a fourth wave
// (six views would spill 60 bytes and more: left alone).
// (float arithmetic; in double the registers are left to the compiler)
constexpr int forward_min_waves(int lpp, int nv, int corr, int reduce, bool wide_real) {
  if (wide_real) return 1;
  if (reduce != 0 && corr <= 1 && nv == 4 && lpp >= 2) return 4;
  if (corr > 1 || reduce != 0) return 1;
  return nv >= 5 ? 4 : (nv >= 3 && lpp == 4) ? 5 : 1;
}

// At most five waves per SIMD: with six (the two-view instantiation needs only 80 VGPRs)
// the waves of a CU evict each other's taps from L1 and the kernel is 6 % slower.  The minimum of three and
// four views of 16 channels likewise with five instead of four (f16, 200 x 260 x 32: 85.8 against 81.6 us).
constexpr int forward_max_waves(int lpp, int nv, int corr, int reduce) {
  return reduce != 0 && corr == 0 && lpp == 4 && nv >= 3 && nv <= 4 ? 4 : 5;
}

// LIT: the mean in the reference's operand order too, every operation rounded by itself, so that the
// result is the plain evaluation's to the bit.  Double is always evaluated that way: the rows are
// twice as long and the stores bound the launch as before (two views, 32 channels, 128 x 160 x 192:
// 1.04 GB in 243 us, 4.3 TB/s; 430 us with a lane per channel, which reads every record and offset
// once for two pixels instead of eight).
// PAD: fewer channels than the pixel's lanes hold (20, 24, 28 on eight lanes), as in the gradient kernel
// below: the lanes past the last channel repeat the last lane's work and store nothing.  Literal, so
// that the results are those of the lane-per-channel kernels, where two pixels share a wave instead of
// eight (24 channels: mean over two views, 89 x 106 x 192, four images 433 -> 255 us; aggregate, six
// views, 130 x 153 x 56, 362 -> 182 us; f16 groups, five views, 111 x 152 x 25, 155 -> 73 us; minimum
// over five views, 63 x 85 x 37, 47 -> 36 us).
template <typename S, int VEC, int LPP, int NV, int CORR, int REDUCE = 0, bool PAD = false,
          bool LIT = (sizeof(S) == 8 || PAD)>
// (waves per SIMD: see forward_min_waves and forward_max_waves)
__global__ __launch_bounds__(64)
__attribute__((amdgpu_waves_per_eu(forward_min_waves(LPP, NV, CORR, REDUCE, sizeof(S) == 8),
                                   forward_max_waves(LPP, NV, CORR, REDUCE)))) void forward_kernel(
    const Args<S> a, const Geometry g) {
  using R = typename Storage<S>::Real;
  using R4 = Four<R>;
  constexpr int PPW = 64 / LPP;
  // bytes of a float4's worth of records per float of lane offset (p4, q4 below)
  constexpr unsigned kR4 = sizeof(R);
  constexpr int GAP = lane_gap(LPP, CORR, (int)sizeof(S), PAD);
  static_assert(!PAD || !best_pair_op(CORR), "CostVolumeV3: whole pixels");
  // Three views and more in double: the views take turns with one set of taps (four sets of four
  // channels are 128 registers), also in the ops that keep a set per view in float.
  constexpr bool kOneSet = sizeof(R) == 8 && NV >= 3 && !best_pair_op(CORR);
  constexpr int NT = kOneSet ? 1 : NV;
  extern __shared__ __align__(16) unsigned char smem[];
  Tile<LPP> t;
  // (one or two views only: the instantiations for more views are held to a register budget
  // that two more live registers break -- f16 cascade forward 95 -> 107 us with them)
  Touched touched{0u, 0u};
  if constexpr (NV <= 2) touched = touch_images(a);
  if (!locate_tile<S, LPP>(a, g, t)) {
    if constexpr (NV <= 2) keep_alive(touched);
    return;
  }
  const int C = PAD ? (int)a.C : VEC * LPP;
  constexpr int kUnit = cell_unit(VEC * LPP, PAD);
  const int D = (int)a.D, N = (int)a.N, srcH = (int)a.srcH, srcW = (int)a.srcW;
  const R half = a.half;
  const bool ch_ok = !PAD || t.cl * VEC < C;
  const int clc = PAD ? min(t.cl, C / VEC - 1) : t.cl;  // the lane whose channels this lane holds
  const int ch0 = lane_first(clc, GAP);
  // LDS records: wts[NV][LPP][PPW] then off[NV][LPP][PPW], addressed as (lane-dependent
  // byte offset) + (compile-time constant) so that the constant lands in the instruction's
  // offset field instead of costing a register per unrolled depth
  constexpr int kWts = 0, kOff = NV * 64 * (int)sizeof(R4), kRec = kOff + NV * 64 * 4;
  const unsigned p4 = (unsigned)t.p * 4u;                 // reader: pixel p
  const unsigned q4 = (unsigned)(t.cl * PPW + t.p) * 4u;  // writer: lane (p, j)

  // (one set: the views' row products, twelve registers each, are computed where a chunk needs them)
  const R ref_w = static_cast<R>(t.w) + half, ref_h = static_cast<R>(t.h) + half;
  Cameras<NT, R> cam;
  if constexpr (!kOneSet) load_cameras<S, NT>(a, t.b, t.view0, ref_w, ref_h, cam);
  const R base = a.depth_grid ? R(0) : a.base_plane[t.pix];
  R ref[VEC];
  if constexpr (CORR != 4) {
    load_vec<S, VEC, false, GAP>(a.ref + t.pix * C + ch0, ref);
    if constexpr (best_pair_op(CORR)) {
      // CostVolumeV3: every lane of a pixel reads all of the pixel's reference groups
      static_assert(!best_pair_op(CORR) || (LPP > 1 && VEC == 4), "CostVolumeV3: wide pixels");
      R *s_ref = reinterpret_cast<R *>(smem + kRec);  // behind the records
#pragma unroll
      for (int c = 0; c < VEC; ++c) s_ref[t.p * (VEC * LPP) + t.cl * VEC + c] = ref[c];
      wave_sync();
    }
  } else {
#pragma unroll
    for (int c = 0; c < VEC; ++c) ref[c] = R(0);  // the warp-only op has no reference image
  }
  constexpr int kWideSub = CORR == 5 ? 2 : 8;  // CostVolumeV3: the wider of the kernel's two group widths
  Two<R> ends{};
  if constexpr (CORR == 5) ends = ref_ends<LPP>(ref);
  const S *view[NV];
#pragma unroll
  for (int n = 0; n < NV; ++n)
    view[n] = a.src + ((int64_t)t.b * N + (n < N ? n : 0)) * srcH * srcW * C;  // (uniform)
  const int row_step = srcW * C;

  constexpr bool kRaw = is_half<S>() && REDUCE == 0 && !LIT;
  Taps<S, VEC, kRaw> tap[NT];
  int cur[NT];
#pragma unroll
  for (int n = 0; n < NT; ++n) cur[n] = -1;

  // CORR: 0 squared difference per channel, 1 group correlation, 2 squared difference
  // summed over all channels (one value per voxel), 4 the samples themselves, one row per
  // (voxel, view), and a 0/1 mask per (voxel, view)
  // (feature_aggregate_kernels_gpu.cu.cc:33-121)
  // 3: CostVolumeV3, per view the largest correlation of any (source group, reference group)
  // pair; MEAN averages the views' maxima, MIN keeps the largest with (view, reference group,
  // source group) as its mask (cost_volume_kernels_gpu_v3.cu.cc:52-146, :148-262)
  const int OC = CORR == 1 ? a.groups : (CORR == 2 || best_pair_op(CORR)) ? 1 : C;
  const int goff = group_offset<VEC>(clc, g.sub);  // first of this lane's group values in a row
  // the cost rows of the per-channel ops (and the sample rows of the warp-only op) stream past
  // the caches where they cover whole lines
  constexpr bool kNtRows = !PAD && whole_lines(VEC * LPP, (int)sizeof(S));
  constexpr bool kAsk = half_lines(LPP, NV, CORR, (int)sizeof(S), PAD);
  const bool stream_halves = kAsk && g.stream_halves;
  // one value per voxel that is added up in channel order
  constexpr bool kRowSums = CORR == 2 && (REDUCE == 1 || LIT);
  const int d_lo = t.d_lo, d_hi = t.d_hi;
  // the cost-map layers' default fill folded into the store: where no view was accepted the
  // scalar is written instead of the cost (custom_layers.py:52-57, :78-83)
  const bool fill = a.default_cost != nullptr;
  const R dflt = fill ? *a.default_cost : R(0);
  // this pixel's output rows (the 64-bit product once per wave, not once per depth)
  S *const out_pix = a.cost + t.pix * D * OC;
  int32_t *const mask_pix = a.mask + t.pix * D * OC;
  for (int d0 = d_lo; d0 < d_hi; d0 += LPP) {
    // ---- phase 1: reprojection by lane (p, j = cl) --------------------------------------
    int r_off[NV];
    R4 r_wts[NV];
    unsigned vmask = 0u;  // views accepted for lane (p, j)'s own voxel
    {
      const int d = d0 + t.cl;
      const bool d_ok = d < d_hi;
      const R depth = d_ok ? voxel_depth(a, t.pix, t.b, d, base) : R(1);
      int cnt = 0;
#pragma unroll
      for (int n = 0; n < NV; ++n) {
        Hit<R> hit;
        if constexpr (kOneSet) load_cameras<S, 1>(a, t.b, n, ref_w, ref_h, cam);
        reproject<NT, R>(cam, kOneSet ? 0 : n, depth, half, g.src_h_max, g.src_w_max, srcW, n < N && d_ok, hit);
        const int off = PAD && hit.cell >= 0 ? hit.cell * C : hit.cell;
        cnt += off >= 0;
        if constexpr (kRowSums) vmask |= (off >= 0 ? 1u : 0u) << n;
        if constexpr (CORR == 4) {
          if (n < N && d_ok && t.pix_ok)
            a.mask[(t.pix * D + d) * N + n] = off >= 0 ? 1 : 0;
        }
        if constexpr (LPP > 1) {
          lds_at<int>(smem, q4, kOff + (n * LPP * PPW) * 4) = off;
          lds_at<R4>(smem, q4 * kR4, kWts + (n * LPP * PPW) * (int)sizeof(R4)) =
              R4{hit.k00, hit.k01, hit.k11, hit.k10};
        } else {
          r_off[n] = off;
          r_wts[n] = R4{hit.k00, hit.k01, hit.k11, hit.k10};
        }
      }
      if constexpr (REDUCE == 0 && CORR != 4)
        if (d_ok && t.pix_ok) a.mask[t.pix * D + d] = cnt;
    }
    if constexpr (LPP > 1) wave_sync();
    if constexpr (kRowSums) {
      // Minimum over the views of the squared difference summed over ALL channels
      // (cost_aggregate_kernels_gpu.cu.cc:128-229).  The mask names the winning view, so the
      // sum has to be the reference's: channel 0 first, every product and sum rounded
      // separately.  View by view, the channel lanes leave the chunk's squares in LDS and the
      // lane that owns voxel (p, d0 + cl) adds its row up in channel order.  The mean in its
      // literal form is one such sum through all accepted views (:33-125).
      constexpr int kSq = kRec;                           // behind the records
      constexpr int ROWB = (VEC * LPP + 4) * (int)sizeof(R);  // bytes per (pixel, depth) row
      R best = REDUCE == 1 ? Limits<R>::max() : R(0);     // numeric_limits<T>::max(), :170
      int win = -1;
#pragma unroll
      for (int n = 0; n < NV; ++n) {
        constexpr int kMany = kOneSet ? 0 : 1;
        Taps<S, VEC, kRaw> &tp = tap[n * kMany];
        int &cur1 = cur[n * kMany];
        if constexpr (kOneSet) cur1 = -1;
        R own[VEC];  // LPP == 1: this lane holds the whole pixel
        constexpr int HALF = squares_depths(LPP, NV, sizeof(R) == 8);  // depths staged together
#pragma unroll
        for (int j0 = 0; j0 < LPP; j0 += HALF) {
        if (j0 > 0 && d0 + j0 >= d_hi) continue;  // (uniform: nothing in the second half)
#pragma unroll
        for (int jj = j0; jj < j0 + HALF; ++jj) {
          if (d0 + jj >= d_hi) {
            if constexpr (LPP >= 16) continue; else break;
          }
          int off;
          R4 wt;
          if constexpr (LPP > 1) {
            off = lds_at<int>(smem, p4, kOff + ((n * LPP + jj) * PPW) * 4);
            wt = lds_at<R4>(smem, p4 * kR4, kWts + ((n * LPP + jj) * PPW) * (int)sizeof(R4));
          } else {
            off = r_off[n];
            wt = r_wts[n];
          }
          R sq[VEC];
#pragma unroll
          for (int c = 0; c < VEC; ++c) sq[c] = R(0);
          if (off >= 0) {
            if (off != cur1) {
              cur1 = off;
              load_cell<S, VEC, GAP, kUnit>(view[n], off, C, row_step, (unsigned)ch0, tp);
            }
#pragma unroll
            for (int c = 0; c < VEC; ++c) {
              const R smp = wt.x * tp(0, c) + wt.y * tp(1, c) + wt.z * tp(2, c) + wt.w * tp(3, c);
              const R diff = smp - ref[c];
              sq[c] = diff * diff;
            }
          }
          if constexpr (LPP > 1) {
            const unsigned own_at = (unsigned)(t.p * HALF * ROWB + ch0 * (int)sizeof(R));
            slot_write<GAP>(&lds_at<R>(smem, own_at, kSq + (jj - j0) * ROWB), sq);
          } else {
#pragma unroll
            for (int c = 0; c < VEC; ++c) own[c] = sq[c];
          }
        }
        if constexpr (LPP > 1) wave_sync();
        if (((vmask >> n) & 1u) && (HALF == LPP || (unsigned)(t.cl - j0) < (unsigned)HALF)) {
          R tot = REDUCE == 1 ? R(0) : best;
          if constexpr (LPP > 1) {
#pragma unroll
            for (int k = 0; k < LPP; ++k) {
              if (PAD && k * VEC >= C) continue;  // (uniform)
              const R4 v = lds_at<R4>(smem, (unsigned)((t.p * HALF + (HALF == LPP ? t.cl : t.cl % HALF)) * ROWB),
                                      kSq + k * VEC * (int)sizeof(R));
              tot += v.x;
              tot += v.y;
              tot += v.z;
              tot += v.w;
            }
          } else {
#pragma unroll
            for (int c = 0; c < VEC; ++c) tot += own[c];
          }
          if constexpr (REDUCE == 0) best = tot;
          else if (best > tot) best = tot, win = n;  // strict: the earliest view keeps a tie (:217)
        }
        if constexpr (LPP > 1) wave_sync();
        }  // half of the chunk
      }
      const int d = d0 + t.cl;
      if (d < d_hi && t.pix_ok) {
        R out = dflt;
        if constexpr (REDUCE == 1) {
          if (win >= 0) out = best / static_cast<R>(C);  // :222-227
          a.mask[t.pix * D + d] = win;
        } else {
          if (vmask != 0u) out = best / static_cast<R>(__popc(vmask) * C);  // :118-123
        }
        reinterpret_cast<R *>(a.cost)[t.pix * D + d] = out;
      }
      continue;
    }
    if constexpr (CORR == 4 && kOneSet) {
      // the samples alone, view by view (a row per voxel and view: nothing is summed)
#pragma unroll
      for (int n = 0; n < NV; ++n) {
        int cur1 = -1;
#pragma unroll
        for (int jj = 0; jj < LPP; ++jj) {
          if (d0 + jj >= d_hi || n >= N) continue;
          const int off = LPP > 1 ? lds_at<int>(smem, p4, kOff + ((n * LPP + jj) * PPW) * 4) : r_off[n];
          R smp[VEC];
#pragma unroll
          for (int c = 0; c < VEC; ++c) smp[c] = R(0);
          if (off >= 0) {
            R4 wt;
            if constexpr (LPP > 1)
              wt = lds_at<R4>(smem, p4 * kR4, kWts + ((n * LPP + jj) * PPW) * (int)sizeof(R4));
            else
              wt = r_wts[n];
            if (off != cur1) {
              cur1 = off;
              load_cell<S, VEC, GAP, kUnit>(view[n], off, C, row_step, (unsigned)ch0, tap[0]);
            }
#pragma unroll
            for (int c = 0; c < VEC; ++c)
              smp[c] = wt.x * tap[0](0, c) + wt.y * tap[0](1, c) + wt.z * tap[0](2, c) + wt.w * tap[0](3, c);
          }
          if (t.pix_ok && ch_ok)
            store_row<S, VEC, kNtRows, kAsk, GAP>(a.cost + ((t.pix * D + d0 + jj) * N + n) * C + ch0, smp, stream_halves);
        }
      }
      if constexpr (LPP > 1) wave_sync();
      continue;
    }
    if constexpr ((CORR == 0 || CORR == 1) && (NV >= 5 || (NV >= 3 && LPP == 4) || kOneSet)) {
      // ---- phase 2, one view at a time (many views) ---------------------------------------
      // With every view's four taps live at once the kernel needs ~25 registers per view
      // (171 for six views: two waves per SIMD).  Here a block of up to eight depths keeps
      // its accumulators and the views take turns with one set of taps, so the register count
      // hardly depends on the number of views.  Every accumulator still receives the views in
      // order 0..N-1 with the same operations, so the results are those of the
      // depth-by-depth loop.  (Measurements decide where this form is used: for three or four
      // views the depth-by-depth loop needs fewer registers at 32+ channels, and with one or
      // two lanes per pixel its taps, which survive from chunk to chunk, matter more.)
      // (double: blocks of four depths, whose accumulators take the registers of eight in float)
      constexpr int kMostDB = sizeof(R) == 8 ? 4 : 8;
      constexpr int DB = LPP < kMostDB ? LPP : kMostDB;
      // Two views side by side where the registers hold two sets of taps: their gathers are in flight
      // together, and what these kernels do most is wait for them (six wide-baseline views, VALU 45 %, waiting
      // 75 % of the waves' time: 4.6 -> 4.3 ms; 200 x 260 x 96 477 -> 435 us, five views, 128 x 160 x 48, 85.7 ->
      // 80.9; 16 channels, six views, 148 -> 128, four 108 -> 103; minima 2-4 %; f16, five
      // views, 94 -> 88).  Not with taps that are widened, and so waited for, as soon as they are loaded (five
      // views 94 -> 96), nor in double.
      constexpr int VW = (sizeof(S) == 4 || kRaw) && NV % 2 == 0 && LPP >= 4 ? 2 : 1;
      static_assert(NV % VW == 0, "whole groups of views");
      // One view at a time: its arithmetic in the branch that fetched its taps, not in a second one (bf16 groups
      // of four, 64 channels, six views, 63 x 82 x 10, four images: 76 -> 63 us; mean 126 -> 120).  Double is
      // faster with two branches (32 channels, four views, 120 x 160 x 48: 125 against 128; samples 362, 368).
      constexpr bool kOneBranch = VW == 1 && sizeof(R) == 4;
#pragma unroll
      for (int j0 = 0; j0 < LPP; j0 += DB) {
      R acc[DB][VEC];
      int arg[REDUCE == 1 ? DB : 1][VEC];
      int kcnt[DB];
#pragma unroll
      for (int jj = 0; jj < DB; ++jj) {
        kcnt[jj] = 0;
#pragma unroll
        for (int c = 0; c < VEC; ++c) {
          acc[jj][c] = REDUCE == 0 ? R(0) : CORR == 0 ? Limits<R>::max() : Limits<R>::min_positive();
          if constexpr (REDUCE == 1) arg[jj][c] = -1;
        }
      }
#pragma unroll
      for (int n = 0; n < NV; n += VW) {
        int cur1[VW];
        Taps<S, VEC, kRaw> tp[VW];
#pragma unroll
        for (int v = 0; v < VW; ++v) cur1[v] = -1;
#pragma unroll
        for (int jj = 0; jj < DB; ++jj) {
          if (d0 + j0 + jj >= d_hi) continue;
          int off[VW];  // -1 also for a view beyond N (phase 1 leaves those records empty)
          R4 wt[VW];
          auto fetch = [&](int v) __attribute__((always_inline)) {
            if constexpr (LPP > 1)
              wt[v] = lds_at<R4>(smem, p4 * kR4, kWts + (((n + v) * LPP + j0 + jj) * PPW) * (int)sizeof(R4));
            else
              wt[v] = r_wts[n + v];
            if (off[v] != cur1[v]) {
              cur1[v] = off[v];
              load_cell<S, VEC, GAP, kUnit>(view[n + v], off[v], C, row_step, (unsigned)ch0, tp[v]);
            }
          };
          auto add = [&](int v) __attribute__((always_inline)) {
          ++kcnt[jj];
          if constexpr (REDUCE == 1 || LIT) {
            R val[VEC];
#pragma unroll
            for (int c = 0; c < VEC; ++c) {
              const R smp = wt[v].x * tp[v](0, c) + wt[v].y * tp[v](1, c) + wt[v].z * tp[v](2, c) + wt[v].w * tp[v](3, c);
              if (CORR == 0) {
                const R diff = smp - ref[c];
                val[c] = diff * diff;
              } else {
                val[c] = smp * ref[c];
              }
            }
            if (REDUCE == 0 && CORR == 0) {
#pragma unroll
              for (int c = 0; c < VEC; ++c) acc[jj][c] += val[c];
            } else if (REDUCE == 0) {
              add_groups(acc[jj], val, g.sub, t.cl);
            } else if (CORR == 0) {
#pragma unroll
              for (int c = 0; c < VEC; ++c)
                if (acc[jj][c] > val[c]) acc[jj][c] = val[c], arg[jj][c] = n + v;
            } else {
              keep_larger_groups(acc[jj], arg[jj], val, g.sub, t.cl, n + v);
            }
          } else {
#pragma unroll
            for (int c = 0; c < VEC; ++c) {
              if (CORR != 1) {
                R diff = mad(wt[v].x, tp[v](0, c), -ref[c]);
                diff = mad(wt[v].y, tp[v](1, c), diff);
                diff = mad(wt[v].z, tp[v](2, c), diff);
                diff = mad(wt[v].w, tp[v](3, c), diff);
                acc[jj][c] = mad(diff, diff, acc[jj][c]);
              } else {
                R smp = kRaw ? mad(wt[v].x, tp[v](0, c), R(0)) : wt[v].x * tp[v](0, c);
                smp = mad(wt[v].y, tp[v](1, c), smp);
                smp = mad(wt[v].z, tp[v](2, c), smp);
                smp = mad(wt[v].w, tp[v](3, c), smp);
                acc[jj][c] = mad(smp, ref[c], acc[jj][c]);
              }
            }
          }
          };
#pragma unroll
          for (int v = 0; v < VW; ++v) {
            if constexpr (LPP > 1)
              off[v] = lds_at<int>(smem, p4, kOff + (((n + v) * LPP + j0 + jj) * PPW) * 4);
            else
              off[v] = r_off[n + v];
            if (off[v] < 0) continue;
            fetch(v);
            if constexpr (kOneBranch) add(v);
          }
          if constexpr (!kOneBranch) {
#pragma unroll
            for (int v = 0; v < VW; ++v)
              if (off[v] >= 0) add(v);
          }
        }
      }
#pragma unroll
      for (int jj = 0; jj < DB; ++jj) {
        const int d = d0 + j0 + jj;
        if (d >= d_hi || !t.pix_ok || !ch_ok) continue;
        S *out = out_pix + d * OC;  // d * OC is uniform: one add per lane
        if constexpr (REDUCE == 1) {
          int32_t *mout = mask_pix + d * OC;
          if (fill) {
#pragma unroll
            for (int c = 0; c < VEC; ++c)
              if (arg[jj][c] < 0) acc[jj][c] = dflt;
          }
          if (CORR == 0) {
            store_row<S, VEC, kNtRows, kAsk, GAP>(out + ch0, acc[jj], stream_halves);
            store_winners<VEC, LPP, GAP, PAD>(mout + ch0, arg[jj]);
          } else {
            store_groups<S, VEC, LPP, PAD, kAsk>(out + goff, acc[jj], g.sub, stream_halves);
            if (g.sub == 1) store_ints<VEC, !PAD && whole_lines(VEC * LPP, 4)>(mout + goff, arg[jj]);
            else if (g.sub == 2) store_ints<VEC / 2, !PAD && whole_lines(VEC * LPP / 2, 4)>(mout + goff, arg[jj]);
            else if (g.sub == 4 || (t.cl & 1)) store_ints<1, !PAD && whole_lines(VEC * LPP / 4, 4)>(mout + goff, arg[jj]);
          }
        } else {
          mean_of<LIT>(acc[jj], kcnt[jj]);
          if (CORR == 0) {
            if (fill && kcnt[jj] == 0) {
#pragma unroll
              for (int c = 0; c < VEC; ++c) acc[jj][c] = dflt;
            }
            store_row<S, VEC, kNtRows, kAsk, GAP>(out + ch0, acc[jj], stream_halves);
          } else {
            R grp[VEC];
            fold_or_keep<LIT>(acc[jj], g.sub, grp);
            if (fill && kcnt[jj] == 0) {
#pragma unroll
              for (int c = 0; c < VEC; ++c) grp[c] = dflt;
            }
            store_groups<S, VEC, LPP, PAD, kAsk>(out + goff, grp, g.sub, stream_halves);
          }
        }
      }
      }  // block of depths
      if constexpr (LPP > 1) wave_sync();
      continue;
    }
    R agg_out = R(0);
    int v3_out[3] = {-1, -1, -1};
    // ---- phase 2: channel arithmetic by lane (p, channel slice) ---------------------------
#pragma unroll
    for (int jj = 0; jj < LPP; ++jj) {
      const int d = d0 + jj;
      if (d >= d_hi) {
        // (a `break` gives the widest tile a run-time trip count, which keeps the compiler
        // from unrolling it and sends its register arrays to scratch memory)
        if constexpr (LPP >= 16) continue; else break;
      }
      R acc[VEC];
      int arg[VEC];  // REDUCE == 1: winning view per channel (or per group)
#pragma unroll
      for (int c = 0; c < VEC; ++c) {
        // numeric_limits::max() / ::min() seeds, cost_volume_kernels_gpu.cu.cc:174-177 and
        // cost_volume_kernels_gpu_v2.cu.cc:179
        acc[c] = REDUCE == 0 ? R(0) : CORR == 0 ? Limits<R>::max() : Limits<R>::min_positive();
        arg[c] = -1;
      }
      int k = 0;
      R v3_acc = REDUCE == 0 ? R(0) : Limits<R>::min_positive();  // :76, :193
      int v3_view = -1, v3_code = 0;
#pragma unroll
      for (int n = 0; n < NT; ++n) {
        int off;
        R4 wt;
        if constexpr (LPP > 1) {
          off = lds_at<int>(smem, p4, kOff + ((n * LPP + jj) * PPW) * 4);
          wt = lds_at<R4>(smem, p4 * kR4, kWts + ((n * LPP + jj) * PPW) * (int)sizeof(R4));
        } else {
          off = r_off[n];
          wt = r_wts[n];
        }
        if constexpr (best_pair_op(CORR)) {
          if (off >= 0) {
            if (off != cur[n]) {
              cur[n] = off;
              load_cell<S, VEC, GAP, kUnit>(view[n], off, C, row_step, (unsigned)ch0, tap[n]);
            }
            R smp[VEC];
#pragma unroll
            for (int c = 0; c < VEC; ++c)
              smp[c] = wt.x * tap[n](0, c) + wt.y * tap[n](1, c) + wt.z * tap[n](2, c) +
                       wt.w * tap[n](3, c);
            const R *ref_row = reinterpret_cast<const R *>(smem + kRec) + t.p * (VEC * LPP);
            R best;
            int code;
            if (g.sub == kWideSub)
              v3_best_pair<R, VEC, LPP, kWideSub, REDUCE == 1>(smp, ref_row, ends, t.cl, best, code);
            else
              v3_best_pair<R, VEC, LPP, kWideSub / 2, REDUCE == 1>(smp, ref_row, ends, t.cl, best, code);
            if constexpr (REDUCE == 0) {
              v3_acc += best;  // the seed when no pair exceeds it (:113-131)
            } else if (v3_acc < best) {
              // one running maximum over views and pairs (:231-250)
              v3_acc = best, v3_view = n, v3_code = code;
            }
            ++k;
          }
          continue;
        }
        if constexpr (CORR == 4) {
          // the sample in the reference's operand order (bit-identical to the plain
          // evaluation), zeros for a view that is not accepted
          R smp[VEC];
#pragma unroll
          for (int c = 0; c < VEC; ++c) smp[c] = R(0);
          if (off >= 0) {
            if (off != cur[n]) {
              cur[n] = off;
              load_cell<S, VEC, GAP, kUnit>(view[n], off, C, row_step, (unsigned)ch0, tap[n]);
            }
#pragma unroll
            for (int c = 0; c < VEC; ++c)
              smp[c] = wt.x * tap[n](0, c) + wt.y * tap[n](1, c) + wt.z * tap[n](2, c) +
                       wt.w * tap[n](3, c);
          }
          if (n < N && t.pix_ok && ch_ok)
            store_row<S, VEC, kNtRows, kAsk, GAP>(a.cost + ((t.pix * D + d) * N + n) * C + ch0, smp, stream_halves);
          continue;
        }
        if (off >= 0) {
          if (off != cur[n]) {
            cur[n] = off;
            load_cell<S, VEC, GAP, kUnit>(view[n], off, C, row_step, (unsigned)ch0, tap[n]);
          }
          if constexpr (REDUCE == 1 || LIT) {
            R val[VEC];
#pragma unroll
            for (int c = 0; c < VEC; ++c) {
              const R smp = wt.x * tap[n](0, c) + wt.y * tap[n](1, c) + wt.z * tap[n](2, c) +
                            wt.w * tap[n](3, c);
              if (CORR != 1) {
                const R diff = smp - ref[c];
                val[c] = diff * diff;
              } else {
                val[c] = smp * ref[c];
              }
            }
            if (REDUCE == 0 && CORR != 1) {
#pragma unroll
              for (int c = 0; c < VEC; ++c) acc[c] += val[c];
            } else if (REDUCE == 0) {
              add_groups(acc, val, g.sub, t.cl);
            } else if (CORR == 0) {
#pragma unroll
              for (int c = 0; c < VEC; ++c)
                if (acc[c] > val[c]) acc[c] = val[c], arg[c] = n;
            } else {
              keep_larger_groups(acc, arg, val, g.sub, t.cl, n);
            }
            ++k;
            continue;
          }
#pragma unroll
          for (int c = 0; c < VEC; ++c) {
            if (CORR != 1) {
              // sample - ref as one chain of fused multiply-adds
              R diff = mad(wt.x, tap[n](0, c), -ref[c]);
              diff = mad(wt.y, tap[n](1, c), diff);
              diff = mad(wt.z, tap[n](2, c), diff);
              diff = mad(wt.w, tap[n](3, c), diff);
              acc[c] = mad(diff, diff, acc[c]);
            } else {
              R smp = kRaw ? mad(wt.x, tap[n](0, c), R(0)) : wt.x * tap[n](0, c);
              smp = mad(wt.y, tap[n](1, c), smp);
              smp = mad(wt.z, tap[n](2, c), smp);
              smp = mad(wt.w, tap[n](3, c), smp);
              acc[c] = mad(smp, ref[c], acc[c]);
            }
          }
          ++k;
        }
      }
      if constexpr (CORR == 4) continue;  // every view's row is already stored
      if constexpr (best_pair_op(CORR)) {
        // the lane whose slice index equals the depth's place in the chunk keeps the voxel
        if (t.cl == jj) {
          if constexpr (REDUCE == 0) {
            agg_out = k > 0 ? v3_acc / static_cast<R>(k) : R(0);  // :136-141
          } else {
            agg_out = v3_view >= 0 ? v3_acc : R(0);  // :253-257
            v3_out[0] = v3_view;
            v3_out[1] = v3_view >= 0 ? v3_code % kPairRow : -1;
            v3_out[2] = v3_view >= 0 ? v3_code / kPairRow : -1;
          }
        }
        continue;
      }
      if constexpr (REDUCE == 1) {
        if (fill) {
#pragma unroll
          for (int c = 0; c < VEC; ++c)
            if (arg[c] < 0) acc[c] = dflt;
        }
        if (t.pix_ok && ch_ok) {
          S *out = out_pix + d * OC;  // d * OC is uniform: one add per lane
          int32_t *mout = mask_pix + d * OC;
          if (CORR == 0) {
            store_row<S, VEC, kNtRows, kAsk, GAP>(out + ch0, acc, stream_halves);
            store_winners<VEC, LPP, GAP, PAD>(mout + ch0, arg);
          } else {
            store_groups<S, VEC, LPP, PAD, kAsk>(out + goff, acc, g.sub, stream_halves);
            if (g.sub == 1) store_ints<VEC, !PAD && whole_lines(VEC * LPP, 4)>(mout + goff, arg);
            else if (g.sub == 2) store_ints<VEC / 2, !PAD && whole_lines(VEC * LPP / 2, 4)>(mout + goff, arg);
            else if (g.sub == 4 || (t.cl & 1)) store_ints<1, !PAD && whole_lines(VEC * LPP / 4, 4)>(mout + goff, arg);
          }
        }
        continue;
      }
      if constexpr (CORR == 2) {
        // one value per voxel: the pixel's lanes add up their channels; the lane whose
        // slice index equals the depth's place in the chunk keeps the result, so that the
        // chunk is stored as LPP consecutive floats per pixel
        R tot = group_sum<LPP>((acc[0] + acc[1]) + (acc[2] + acc[3]));
        tot = k > 0 ? tot / static_cast<R>(k * C) : dflt;
        if constexpr (LPP > 1) {
          if (t.cl == jj) agg_out = tot;
        } else {
          if (t.pix_ok) reinterpret_cast<R *>(a.cost)[t.pix * D + d] = tot;
        }
        continue;
      }
      mean_of<LIT>(acc, k);
      if (t.pix_ok && ch_ok) {
        S *out = out_pix + d * OC;  // d * OC is uniform: one add per lane
        if (CORR == 0) {
          if (fill && k == 0) {
#pragma unroll
            for (int c = 0; c < VEC; ++c) acc[c] = dflt;
          }
          store_row<S, VEC, kNtRows, kAsk, GAP>(out + ch0, acc, stream_halves);
        } else {
          R grp[VEC];
          fold_or_keep<LIT>(acc, g.sub, grp);
          if (fill && k == 0) {
#pragma unroll
            for (int c = 0; c < VEC; ++c) grp[c] = dflt;
          }
          store_groups<S, VEC, LPP, PAD, kAsk>(out + goff, grp, g.sub, stream_halves);
        }
      }
    }
    if constexpr ((CORR == 2 || best_pair_op(CORR)) && LPP > 1) {
      if (t.pix_ok && d0 + t.cl < d_hi)
        reinterpret_cast<R *>(a.cost)[t.pix * D + d0 + t.cl] = agg_out;
    }
    if constexpr (best_pair_op(CORR) && REDUCE == 1) {
      if (t.pix_ok && d0 + t.cl < d_hi) {
        int32_t *m = a.mask + (t.pix * D + d0 + t.cl) * 3;
        m[0] = v3_out[0], m[1] = v3_out[1], m[2] = v3_out[2];
      }
    }
    if constexpr (LPP > 1) wave_sync();
  }
  if constexpr (NV <= 2) keep_alive(touched);
}

// =========================================================================================
// Backward
// =========================================================================================
// Per-view scatter window: a ring buffer of ROWS x COLS texels (C fp32 sums each) addressed
// by the low bits of the texel coordinates.  `oy, ox` is the window origin: the window
// holds exactly the texels [oy, oy+ROWS) x [ox, ox+COLS).  Because the slot of a texel
// depends only on its coordinates, the four slots of a cell are computed once, by the lane
// that reprojects the voxel, and travel with the record.
// The forms of the window: left to the tile's shape, or fixed by the kernel that owns it.
enum { kNotEight = 0, kEightWide = 1, kEightTall = 2 };  // backward_kernel's EIGHT
enum { kPlainWindow = 0, kSixRows = 6, kFourRows = 4, kSixColumns = 8 };
template <int VEC, int LPP, int FORM = kPlainWindow>
struct Window {
  static constexpr int PPW = 64 / LPP;
  // twice the tile's height by twice its width, at least eight each way: room for the
  // samples' drift in either direction (8 x 8 against 4 x 16 for the 2 x 4 pixels of 32
  // channels: 357 -> 338 us on the MVSNet-stage workload)
  static constexpr int TH = tile_rows(PPW), TW = PPW / TH;
  // kSixRows (eight lanes per pixel, 32 channels, 2 x 4 pixels, kernels held to four waves per
  // SIMD: see backward_waves): six rows instead of eight.  With a 6 KB window the workgroup's
  // LDS is 10 KB, so that sixteen workgroups fit a CU; four rows measured 2 % slower than eight
  // at equal occupancy, six sit between.  The ring index of a row is then a remainder, not a
  // mask.
  // Sixteen lanes per pixel (64 channels, 2 x 2 pixels): a slot is 256 bytes, and with eight rows
  // the window alone held a CU to seven workgroups (20.5 KB each).  Four rows (12.5 KB) let
  // thirteen in; together with the slimming of lean_backward the gradients run three waves
  // per SIMD instead of two (group correlation, four views, 254 x 319 x 16, training pass 2.68
  // -> 1.61 ms; warped features, four views, 73 x 96 x 161: 1218 -> 1045 us).
  // Double doubles a slot: kFourRows for eight lanes per pixel.
  static constexpr int ROWS = FORM == kSixRows                 ? 6
                              : FORM == kFourRows || LPP == 16 ? 4
                                                               : (2 * TH > 8 ? 2 * TH : 8);
  // kSixColumns: the same turned by ninety degrees, for a tile of 4 x 2 pixels.
  static constexpr int COLS = FORM == kSixColumns ? 6 : (2 * TW > 8 ? 2 * TW : 8);
  static constexpr int SLOTS = ROWS * COLS;
  // place of image row / column `i` (not negative) in a ring of LEN
  template <int LEN>
  static __device__ __forceinline__ int ring(unsigned i) {
    if constexpr ((LEN & (LEN - 1)) == 0) {
      return (int)(i & (unsigned)(LEN - 1));
    } else {
      // (i / 6 for every i up to 32769; a general division by a constant takes the high half of a
      // product, four times the issue time of a 24-bit one)
      static_assert(LEN == 6, "the reciprocal below");
      return (int)(i - (__umul24(i, 10923u) >> 16) * 6u);
    }
  }
  // the place after `r`
  template <int LEN>
  static __device__ __forceinline__ int ring_next(int r) {
    if constexpr ((LEN & (LEN - 1)) == 0) return (r + 1) & (LEN - 1);
    else return r == LEN - 1 ? 0 : r + 1;
  }
  static __device__ __forceinline__ int ring_row(unsigned fh) { return ring<ROWS>(fh); }
  static __device__ __forceinline__ int ring_col(unsigned fw) { return ring<COLS>(fw); }
  // image row / column at place `r` of a ring whose window starts at `o` (any sign)
  template <int LEN>
  static __device__ __forceinline__ int unring(int r, int o) {
    if constexpr ((LEN & (LEN - 1)) == 0) {
      return o + ((r - o) & (LEN - 1));
    } else {
      const int first = o >= 0 ? o % LEN : (LEN - 1) - (-1 - o) % LEN;  // (o is uniform)
      const int m = r - first;
      return o + (m < 0 ? m + LEN : m);
    }
  }
  static __device__ __forceinline__ int image_row(int ry, int oy) { return unring<ROWS>(ry, oy); }
  static __device__ __forceinline__ int image_col(int rx, int ox) { return unring<COLS>(rx, ox); }
  static constexpr int C = VEC * LPP;
  static constexpr int STRIDE = C;      // one slot = C consecutive words: 16-byte lane accesses
  static constexpr int kNone = 0x3fffffff;
  static constexpr bool kPacked = SLOTS <= 256;  // four slot numbers fit one word
  static constexpr int kInside = (int)0x80000000u;  // flag in the key word: cell lies in the window

  // slots of the taps 00, 01, 11, 10 of the cell in row `fh` (ring row r0) and column `fw`, one byte each
  static __device__ __forceinline__ unsigned pack_slots(int r0, int r1, unsigned fw) {
    const unsigned rx0 = (unsigned)ring_col(fw), rx1 = (unsigned)ring_next<COLS>((int)rx0);
    const unsigned ry0 = (unsigned)(r0 * COLS), ry1 = (unsigned)(r1 * COLS);
    // bytes: rx0, rx1, rx1, rx0 plus ry0, ry0, ry1, ry1 (v_perm_b32: selectors 0-3 take the second operand's bytes)
    return __builtin_amdgcn_perm(rx1, rx0, 0x00040400u) + __builtin_amdgcn_perm(ry1, ry0, 0x04040000u);
  }
  // whole cell inside the window at origin (oy, ox)?
  static __device__ __forceinline__ bool inside(int key, int oy, int ox) {
    const int fh = (key >> 16) & 0x7fff, fw = key & 0xffff;
    return (unsigned)(fh - oy) < (unsigned)(ROWS - 1) && (unsigned)(fw - ox) < (unsigned)(COLS - 1);
  }
};

// Pixels of up to this many lanes update the scatter window in claimed tap-by-tap rounds
// (see window_add), which needs one claim word per window slot.
constexpr int kClaimLanes = 8;
// ... and from two lanes on the claim words also say which slots hold something: negative where nothing was
// added since the window last let go of the slot (window_move, tagged_rows).  With one lane per pixel a
// pixel would write all four by itself (minimum of CostAggregate, three views of 4 channels, 256 x 320 x 32: 123 -> 130 us).
constexpr bool tagged_slots(int lpp) { return lpp >= 2 && lpp <= kClaimLanes; }

// LDS bytes of the backward kernel: the records of one chunk
//   Four wts, dwt [NV*64] | int2 cell {slots, key|inside} [NV*64] | int off [NV*64] |
//   R scale [64] | R dst [64] (per-voxel depth gradients and CostVolumeV3)
// then the list of texels leaving a window, then the windows.  With one view per workgroup
// the list shares the record space: a window that moves for a chunk as a whole does so before the
// chunk's records are written.  One that follows the runs inside a chunk (end_spread_runs) has a list of
// its own, backward_list_bytes.
// The slim form (double, slim_double) keeps one Four {dh, dw, d sh / d depth, d sw / d depth} for both
// sets of weights, which the lanes expand where a depth starts (eleven operations): 64 bytes less
// per voxel.
template <typename R, int VEC, int LPP, int NV, int FORM = kPlainWindow, bool SLIM = false, bool DST = true>
constexpr int backward_record_bytes() {
  using WN = Window<VEC, LPP, FORM>;
  const int fours = SLIM ? 1 : 2;
  const int rec = LPP > 1 ? NV * 64 * (fours * 4 * (int)sizeof(R) + 12) + (DST ? 2 : 1) * 64 * (int)sizeof(R) : 0;
  const int list = WN::SLOTS * 8;
  const int b = NV == 1 ? (rec > list ? rec : list) : rec + list;
  return (b + 31) / 32 * 32;
}
// The list of a window move between two depths of a chunk, whose records are in use then.
template <typename R, int VEC, int LPP, int FORM = kPlainWindow>
constexpr int backward_list_bytes() {
  using WN = Window<VEC, LPP, FORM>;
  return LPP > 1 && WN::SLOTS * 8 > 4 * WN::C * (int)sizeof(R) ? WN::SLOTS * 8 : 0;
}
template <typename R, int VEC, int LPP, int NV, int FORM = kPlainWindow, bool SLIM = false, bool DST = true>
constexpr int backward_lds_bytes() {
  using WN = Window<VEC, LPP, FORM>;
  // records (or list), windows, one cell (4 texels x C) staged on its way to memory, and for
  // narrow pixels one claim word per window slot
  // and, where that cell's place is too small for it, the list of a move inside a chunk
  return backward_record_bytes<R, VEC, LPP, NV, FORM, SLIM, DST>() +
         (NV * WN::SLOTS * WN::STRIDE + 4 * WN::C) * (int)sizeof(R) +
         (LPP <= kClaimLanes ? WN::SLOTS * 4 : 0) + backward_list_bytes<R, VEC, LPP, FORM>();
}

// The box around the cells of the active lanes of a wave (at least one): `lo` and `hi` hold a lane's smallest
// and largest row and column, packed like a key, kNoLow and kNoHigh for a lane without a cell.  Rows and columns
// are reduced together, in 16-bit halves, by DPP moves within and then across the rows of 16 lanes: 26
// instructions, where four 32-bit reductions took 88 -- a spread sweep makes a box at nearly every depth.
constexpr int kNoLow = 0x7fff7fff, kNoHigh = 0;
typedef short i16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ int min_halves(int a, int b) {
  return __builtin_bit_cast(int, __builtin_elementwise_min(__builtin_bit_cast(i16x2, a), __builtin_bit_cast(i16x2, b)));
}
__device__ __forceinline__ int max_halves(int a, int b) {
  return __builtin_bit_cast(int, __builtin_elementwise_max(__builtin_bit_cast(i16x2, a), __builtin_bit_cast(i16x2, b)));
}
template <int CTRL, int ROWS>
__device__ __forceinline__ void box_step(int &lo, int &hi) {
  int l, h;
  if constexpr (ROWS == 0xf) {  // (every lane reads one: what the register held before is of no interest)
    l = __builtin_amdgcn_mov_dpp(lo, CTRL, 0xf, 0xf, true), h = __builtin_amdgcn_mov_dpp(hi, CTRL, 0xf, 0xf, true);
  } else {
    l = __builtin_amdgcn_update_dpp(lo, lo, CTRL, ROWS, 0xf, false);
    h = __builtin_amdgcn_update_dpp(hi, hi, CTRL, ROWS, 0xf, false);
  }
  lo = min_halves(lo, l), hi = max_halves(hi, h);
}
struct Box {
  int y0, x0, y1, x1;  // first row and column of the cells, last ones of their texels (uniform)
};
__device__ __forceinline__ Box wave_box(int lo, int hi) {
  box_step<0xB1, 0xf>(lo, hi);   // quad_perm 1,0,3,2
  box_step<0x4E, 0xf>(lo, hi);   // quad_perm 2,3,0,1
  box_step<0x141, 0xf>(lo, hi);  // row_half_mirror
  box_step<0x140, 0xf>(lo, hi);  // row_mirror
  box_step<0x142, 0xa>(lo, hi);  // row_bcast15 into rows 1 and 3
  box_step<0x143, 0xc>(lo, hi);  // row_bcast31 into rows 2 and 3: lane 63 has everything
  const int l = __builtin_amdgcn_readlane(lo, 63), h = __builtin_amdgcn_readlane(hi, 63);
  return Box{l >> 16, l & 0xffff, (h >> 16) + 1, (h & 0xffff) + 1};
}

// Adds to element `e` of a view's image, whose 2^29 elements at most (make_plan) are addressed as the
// view's uniform base plus 32 bits of bytes.
template <typename R>
__device__ __forceinline__ void atomic_at(R *image, unsigned e, R v) {
  atomic_add(reinterpret_cast<R *>(reinterpret_cast<char *>(image) + e * (unsigned)sizeof(R)), v);
}

// Moves the window of one view to origin (ny, nx): every texel that was added to and falls outside the new
// window is written out with dense global atomics (C consecutive floats per texel, 64/C texels per
// instruction, UN instructions per round: their LDS reads go out together) and its slot is cleared.
// Uniform control flow.  `tags`: see tagged_slots.  A spread sweep leaves some fifteen of the 48 or 64 slots at a
// time; with the empty ones left out, the list holding offsets instead of indices and the box of wave_box six
// wide-baseline views, 288 x 384 x 128, take 10.5 ms instead of 11.6.  `cm`:
// channels of a texel in memory (a slot may be padded; padding stays zero and is never written out).
template <int VEC, int LPP, int FORM = kPlainWindow, int UN = 4, typename R>
__device__ __forceinline__ void window_move(int &oy, int &ox, int ny, int nx, R *data, int *tags,
                                            int *list, R *gview, int srcW, int lane, int cm) {
  using WN = Window<VEC, LPP, FORM>;
  if (oy != WN::kNone) {
    wave_sync();  // the adds of the chunk before are complete and visible
    int count = 0;
    for (int sb = 0; sb < WN::SLOTS; sb += 64) {
      const int s = sb + lane;  // (a window of 48 slots: the last lanes have none)
      const int ry = s / WN::COLS, rx = s % WN::COLS;
      const int y = WN::image_row(ry, oy), x = WN::image_col(rx, ox);
      bool leaving = s < WN::SLOTS && !((unsigned)(y - ny) < (unsigned)WN::ROWS &&
                                        (unsigned)(x - nx) < (unsigned)WN::COLS);
      if constexpr (tagged_slots(LPP)) leaving = leaving && tags[s] >= 0;
      const unsigned long long m = __ballot(leaving);
      if (leaving) {
        const int rank = count + (int)__builtin_amdgcn_mbcnt_hi(
            (unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));  // leaving lanes below me
        list[2 * rank] = s * WN::STRIDE;
        list[2 * rank + 1] = (y * srcW + x) * cm;
        if constexpr (tagged_slots(LPP)) tags[s] = -1;
      }
      count += __popcll(m);
    }
    if (count > 0) {
      wave_sync();
      constexpr int EPI = 64 / WN::C;  // texels per instruction
      const int sub_e = lane / WN::C, j = lane - sub_e * WN::C;
      const int2 *pairs = reinterpret_cast<const int2 *>(list);
      for (int e0 = 0; e0 < count; e0 += UN * EPI) {
        int2 le[UN];
        R v[UN];
#pragma unroll
        for (int u = 0; u < UN; ++u) le[u] = pairs[min(e0 + u * EPI + sub_e, count - 1)];
#pragma unroll
        for (int u = 0; u < UN; ++u) v[u] = data[le[u].x + j];
#pragma unroll
        for (int u = 0; u < UN; ++u) {
          if (e0 + u * EPI + sub_e < count && v[u] != R(0)) {
            data[le[u].x + j] = R(0);
            atomic_at(gview, (unsigned)le[u].y + (unsigned)j, v[u]);
          }
        }
      }
      wave_sync();
    }
  }
  oy = ny;
  ox = nx;
}

// Bitwise OR over the 64 lanes, in registers.
__device__ __forceinline__ unsigned wave_or(unsigned v) {
  v |= (unsigned)__builtin_amdgcn_update_dpp((int)v, (int)v, 0xB1, 0xf, 0xf, false);
  v |= (unsigned)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x4E, 0xf, 0xf, false);
  v |= (unsigned)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x141, 0xf, 0xf, false);
  v |= (unsigned)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x140, 0xf, 0xf, false);
  return (unsigned)__builtin_amdgcn_readlane((int)v, 0) | (unsigned)__builtin_amdgcn_readlane((int)v, 16) |
         (unsigned)__builtin_amdgcn_readlane((int)v, 32) | (unsigned)__builtin_amdgcn_readlane((int)v, 48);
}

// The ring rows of a window that hold something: those with a tag that is not negative (uniform).
template <int VEC, int LPP, int FORM>
__device__ __forceinline__ unsigned tagged_rows(const int *tags, int lane) {
  using WN = Window<VEC, LPP, FORM>;
  unsigned rows = 0u;
#pragma unroll
  for (int sb = 0; sb < WN::SLOTS; sb += 64) {
    const int s = sb + lane;
    const bool held = s < WN::SLOTS && tags[s] >= 0;
    if constexpr (64 % WN::COLS == 0) {
      const unsigned long long m = __ballot(held);
#pragma unroll
      for (int r = 0; r < 64 / WN::COLS; ++r)
        rows |= (m >> (r * WN::COLS) & ((1ull << WN::COLS) - 1ull) ? 1u : 0u) << (sb / WN::COLS + r);
    } else {
      rows |= wave_or(held ? 1u << (s / WN::COLS) : 0u);
    }
  }
  return rows;
}

// Writes out everything a window holds, when its view is done: row by row of the ring
// buffer, and only the rows that hold something, or that some accepted cell of this view ever
// mapped to (`rows`: bit r set when a cell used ring row r; a short sweep over few hypotheses touches three or four
// of the eight, and the untouched ones need neither their LDS reads nor their address
// arithmetic).  All LDS reads of a row are issued together, then its atomics.
template <int VEC, int LPP, int FORM = kPlainWindow, typename R>
__device__ __forceinline__ void window_flush_all(int oy, int ox, const R *data, R *gview,
                                                 int srcW, int lane, unsigned rows, int cm) {
  using WN = Window<VEC, LPP, FORM>;
  if (oy == WN::kNone) return;
  wave_sync();  // the last adds are complete and visible
  constexpr int C = WN::C;
  constexpr int PER_ROW = WN::COLS * C / 64;  // instructions of 64 consecutive floats per row
  static_assert(WN::COLS * C % 64 == 0, "whole instructions per window row");
  if (__popc(rows) > WN::ROWS * 5 / 8) {
    // (nearly) every row in use, as after a long sweep: the whole window in batches of 32
    // instructions whose LDS reads go out together, so that the wave waits for the LDS once
    // per batch instead of once per row (315 against 325 us on the MVSNet-stage workload)
    constexpr int NI = WN::SLOTS * C / 64;
    constexpr int MOST = sizeof(R) == 4 ? 32 : NI % 16 == 0 ? 16 : 8;
    constexpr int BATCH = NI < MOST ? NI : MOST;
    static_assert(NI % BATCH == 0, "whole batches");
#pragma unroll 1
    for (int i0 = 0; i0 < NI; i0 += BATCH) {
      R v[BATCH];
#pragma unroll
      for (int u = 0; u < BATCH; ++u) v[u] = data[(i0 + u) * 64 + lane];
#pragma unroll
      for (int u = 0; u < BATCH; ++u) {
        const int e = (i0 + u) * 64 + lane;  // float index inside the window
        const int sl = e / C, ch = e - sl * C;
        const int ry = sl / WN::COLS, rx = sl - ry * WN::COLS;
        const int y = WN::image_row(ry, oy), x = WN::image_col(rx, ox);
        if (v[u] != R(0)) atomic_at(gview, (unsigned)(y * srcW + x) * (unsigned)cm + (unsigned)ch, v[u]);
      }
    }
    return;
  }
#pragma unroll 1
  for (int ry = 0; ry < WN::ROWS; ++ry) {
    if (!((rows >> ry) & 1u)) continue;  // uniform
    const int y = WN::image_row(ry, oy);
    R v[PER_ROW];
#pragma unroll
    for (int u = 0; u < PER_ROW; ++u) v[u] = data[(ry * PER_ROW + u) * 64 + lane];
#pragma unroll
    for (int u = 0; u < PER_ROW; ++u) {
      const int e = u * 64 + lane;  // float index inside the row
      const int rx = e / C, ch = e - rx * C;
      const int x = WN::image_col(rx, ox);
      // (a slot that was never added to holds zero: texels outside the image never are)
      if (v[u] != R(0)) atomic_at(gview, (unsigned)(y * srcW + x) * (unsigned)cm + (unsigned)ch, v[u]);
    }
  }
}

// The source gradient of one channel of a lane, summed over an open run: taps 00, 01, 11, 10.
// Four adjacent registers: an accumulator of the matrix cores (see the depth loop).
// (matrix accumulators; elsewhere four values of their own)
typedef float f32x4 __attribute__((ext_vector_type(4)));
template <typename R>
struct LooseSums {
  R v[4];
  __device__ __forceinline__ R &operator[](int k) { return v[k]; }
};
// The sum of tap `k` and channel `c` on top of `old`.  As many sums as channels: the channel's own.  Fewer
// (group correlation): the sum of the channel's group, times the channel's reference value.
template <int VEC, int NS, typename R, typename T>
__device__ __forceinline__ R add_tap_sum(R old, T (&v)[NS], const R (&ref)[VEC], int c, int k) {
  if constexpr (NS == VEC) return old + v[c][k];
  else return mad(ref[c], v[c * NS / VEC][k], old);
}

// Adds the four tap images of a finished run into the window (its cell lies inside: one that sticks out
// never gets here, flush_cells_to_memory has taken it).  Called from divergent code by all
// LPP lanes of every pixel whose run just ended.  Float LDS atomics cost about three cycles
// per lane, so the window sums are updated with plain 16-byte read-add-write.  Cells of
// different pixels overlap (a texel is tap 01 of one cell and tap 00 of its neighbour).
// Up to kClaimLanes lanes per pixel (8 to 64 pixels per wave, from two to a dozen firing at
// once): all firing pixels add tap 00, then all tap 01, ... — two pixels then collide only
// if they are on the SAME cell, and those are told apart by a claim: every pending pixel
// writes its number into the claim word of its first texel's slot and the one that reads its
// own number back goes ahead; the others try again (`tags`: one word per slot).  A pixel that
// fires alone skips all that.  Against one pixel per round this takes the headline backward
// from 429 to 400 us; against LDS atomics it halved the time of the 8-channel workloads.
// 16 lanes per pixel (four pixels per wave): the pixels that fire in the same instruction
// take turns, one pixel per round with its four taps in flight together.
template <int VEC, int LPP, bool LEAN = false, int FORM = kPlainWindow, int GAP = 2, int NS, typename R, typename T>
__device__ __forceinline__ void window_add(unsigned slots, int key, T (&v)[NS], const R (&ref)[VEC], R *data,
                                           int *tags, int lane, int cl) {
  using WN = Window<VEC, LPP, FORM>;
  int slot[4];
  if constexpr (WN::kPacked) {
    slot[0] = slots & 255u, slot[1] = (slots >> 8) & 255u, slot[2] = (slots >> 16) & 255u, slot[3] = slots >> 24;
  } else {
    const int fh = (key >> 16) & 0x7fff, fw = key & 0xffff;
    const int ry0 = WN::ring_row((unsigned)fh) * WN::COLS, ry1 = WN::ring_row((unsigned)fh + 1u) * WN::COLS;
    const int rx0 = WN::ring_col((unsigned)fw), rx1 = WN::ring_col((unsigned)fw + 1u);
    slot[0] = ry0 + rx0, slot[1] = ry0 + rx1, slot[2] = ry1 + rx1, slot[3] = ry1 + rx0;
  }
  unsigned char *const base = reinterpret_cast<unsigned char *>(data + lane_first(cl, GAP));
  R *texel[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) texel[k] = reinterpret_cast<R *>(base + slot[k] * (WN::STRIDE * (int)sizeof(R)));
  auto all_at_once = [&]() __attribute__((always_inline)) {
    R old[4][VEC];
#pragma unroll
    for (int k = 0; k < 4; ++k) slot_read<GAP>(texel[k], old[k]);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
#pragma unroll
      for (int i = 0; i < VEC; ++i) old[k][i] = add_tap_sum(old[k][i], v, ref, i, k);
      slot_write<GAP>(texel[k], old[k]);
    }
  };
  // (one tap after the other; `shared`: the next tap may be the texel another pixel has just updated -- the
  // LDS keeps a wave's operations in order, the compiler is held to it here)
  auto one_by_one = [&](bool shared) __attribute__((always_inline)) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      R old[VEC];
      slot_read<GAP>(texel[k], old);
#pragma unroll
      for (int i = 0; i < VEC; ++i) old[i] = add_tap_sum(old[i], v, ref, i, k);
      slot_write<GAP>(texel[k], old);
      if (shared) wave_sync();
    }
  };
  if constexpr (LPP > kClaimLanes) {
    unsigned long long firing = __ballot(true);
    while (firing) {
      const int lead = __ffsll((long long)firing) - 1;
      firing &= ~(((1ull << LPP) - 1ull) << lead);  // retire this pixel's lanes
      if (lane - cl == lead) all_at_once();
      if (firing) wave_sync();
    }
  } else {
    const int me = lane - cl;  // the same in all lanes of a pixel
    if (__popcll(__ballot(true)) == LPP) {
      // one pixel alone (four of ten events on the headline workload): nothing to collide with, its four
      // taps go in flight together -- or, in a kernel held to a register budget, one after the other
      // (twelve registers less at the kernel's peak)
      if constexpr (LEAN) one_by_one(false);
      else all_at_once();
    } else {
      // (the wave leaves this loop together: a pixel that left it by itself would add after it, beside the others)
      bool pending = true;
      do {
        if (pending) tags[slot[0]] = me;
        wave_sync();
        const bool go = pending && tags[slot[0]] == me;
        if (go) one_by_one(true);
        pending = pending && !go;
      } while (__ballot(pending) != 0ull);
    }
    if constexpr (tagged_slots(LPP)) {  // these four slots hold something now
#pragma unroll
      for (int i = 0; i < (LPP >= 4 ? 1 : 2); ++i) {
        const unsigned k = (unsigned)(cl + i * LPP) & 3u;
        static_assert(WN::kPacked, "slot numbers of a byte");
        tags[(slots >> (k * 8u)) & 255u] = me;
      }
    }
    wave_sync();
  }
#pragma unroll
  for (int i = 0; i < NS; ++i) v[i] = T{R(0), R(0), R(0), R(0)};
}

// Cells that no window position covers (the tile's pixels of one depth further apart than the
// window is wide, on strongly magnified views) go to memory directly.  Uniform control flow:
// `m` has the lane bits of every pixel with such a cell (`mine` for the caller's own lanes).  One pixel
// at a time, its lanes lay the four tap images out in LDS as two rows of two adjacent texels
// and the whole wave adds each row as a dense run of 2*C consecutive floats.  Added lane by
// lane from the registers, each 16-byte chunk of a texel would carry one float per
// instruction, and the atomics cost per chunk, not per float.
template <int VEC, int LPP, int GAP, int NS, typename R, typename T>
__device__ __forceinline__ void flush_cells_to_memory(unsigned long long m, bool mine, int key, T (&v)[NS],
                                                      const R (&ref)[VEC], R *stage, R *gview, int srcW, int lane,
                                                      int cl, int cm) {
  constexpr int C = VEC * LPP;
  while (m) {
    const int lead = __ffsll((long long)m) - 1;
    m &= ~(((1ull << LPP) - 1ull) << lead);
    const int k2 = __builtin_amdgcn_readlane(key, lead);  // the same in all lanes of the pixel
    if (lane - cl == lead) {
      // taps 00, 01 (row fh), then 10, 11 (row fh + 1); v is ordered 00, 01, 11, 10
#pragma unroll
      for (int k = 0; k < 4; ++k)
      {
        R w[VEC];
#pragma unroll
        for (int i = 0; i < VEC; ++i) w[i] = NS == VEC ? v[i * NS / VEC][k] : add_tap_sum(R(0), v, ref, i, k);
        slot_write<GAP>(stage + (k == 2 ? 3 : k == 3 ? 2 : k) * C + lane_first(cl, GAP), w);
      }
    }
    wave_sync();
    const int fh = k2 >> 16, fw = k2 & 0xffff;
    R *row0 = gview + (int64_t)(fh * srcW + fw) * cm;
    R *row1 = row0 + (int64_t)srcW * cm;
#pragma unroll
    for (int f0 = 0; f0 < 2 * C; f0 += 64) {
      const int f = f0 + lane;
      if (f < 2 * C) {
        const R a0 = stage[f], a1 = stage[2 * C + f];
        const int e = f / C * cm + f % C;
        if (a0 != R(0)) atomic_add(row0 + e, a0);
        if (a1 != R(0)) atomic_add(row1 + e, a1);
      }
    }
    wave_sync();
  }
  if (mine) {
#pragma unroll
    for (int i = 0; i < NS; ++i) v[i] = T{R(0), R(0), R(0), R(0)};
  }
}

// Waves per SIMD the register budget is held to.  The kernel is latency-bound (its time
// falls in proportion to the resident waves), so one view per workgroup at three waves
// beats two views at two, and four waves beat three wherever registers and LDS allow them.
// Eight lanes per pixel (32 channels), gradient of the mean squared difference: 161 registers
// left alone.  Held to 128 it spills 80 bytes in the depth loop, so the kernel is slimmed
// first (lean_backward): four upstream rows staged at a time instead of eight (16 registers),
// the records of a depth read where the depth starts instead of one depth ahead (10), the
// four window taps of a pixel that fires alone added one after the other (12) -- 127 registers,
// no scratch.  Those three cost 5 % at three waves per SIMD; with the 10 KB of LDS of the
// six-row window the fourth wave gains 11 % (MVSNet-stage backward 301 -> 277 us).
// Likewise the gradients of CostAggregate (both reduces: 137 -> 117 registers) and of
// FeatureAggregate (149 -> 119).  The MIN / MAX gradients of the per-channel ops, whose mask rows kept them
// at 141-166, keep the winners as lane masks in scalar registers instead (find_won: 120-128, no scratch in
// float): 24 channels, six wide-baseline views, 200 x 260 x 64, 1075 -> 908 us; 32 channels, x 96, 1457 -> 1320, two
// views, 128 x 160 x 96, 208 -> 206; 16 channels, three views, x 48, 282 -> 268, bf16, four, 221 -> 207.  The
// wait for the winners costs up to 6 % where three waves per SIMD hold the whole launch: those keep the
// other form (the launcher).  Not the maximum of 8 channels whose views take turns (52-80 bytes of scratch).
// CostVolumeV3 with groups of four and eight likewise, and since its rows of reference and sample are 2 KB of
// LDS more, with a window of four rows (four_row_pairs): 10.1 instead of 14.3 KB and four waves instead of
// 2.75 per SIMD (32 channels in four groups, two views, 120 x 152 x 64, 188 -> 162 us; five views, x 48, 317
// -> 238; in double, 100 x 130 x 32, 171 -> 141; 16 channels 109 -> 96).  Narrower groups need 143 registers:
// slimmed at three waves with the six-row window (12.2 KB: 237 -> 197 us for groups of two).
// Four lanes per pixel (16 channels), gradients of a mean: 130 registers left alone, 121 lean
// (held to 128 without the slimming they spilled three to five); the window of the 4 x 4 pixel
// tile is 4 KB.  CostAggregate and FeatureAggregate the same (134 -> 117-120; six views, 497 x 700 x 41:
// 3.55 -> 3.11 ms).  Two lanes per pixel (8 channels): 119-125 lean, and 122-128 where the views of
// a tile take turns in the workgroup (VLOOP) -- once the compiler is kept from carrying two
// dozen lane-only values through the view loop (see the barrier at the head of that loop;
// with them the kernels spilled 44-68 bytes around the depth loop and four waves were slower
// than three).  Up to 32 bytes of scratch remain in two of those instantiations, outside the
// depth loop: bf16 group-correlation backward 479 -> 462 us cold, 447 -> 417 us warm.
// Group correlation with the tap sums per group (run_sums): 112-128 registers lean, both reduces.
// Sixteen lanes per pixel (64 channels): slimmed, all of them, to three waves (164-222 registers
// left alone, 132-164 slimmed; LDS holds them to 13 workgroups per CU, see Window::ROWS).
// Double: the slimmed code at two waves per SIMD (taps, tap sums and rows of four channels are 100
// registers before anything else, 182-206 in all), whole records and the six-row window, which fit two waves'
// share of the LDS.  Held to 168 registers for a third wave, with the slim records (slim_double), the cameras'
// row products computed again for every chunk and a window of four rows, the gradients that stream
// upstream rows spill 76-130 bytes around the depth loop, and a reload from scratch waits for the
// rows requested before it: 32 channels, two views, 128 x 160 x 192: 745 us against 532 (lane per
// channel: 940), minimum over three views x 64 751 against 372 (673).  CostAggregate has no rows and
// does not spill: three views, 149 x 220 x 116, 524 against 584 us (1460); 64 channels, where LDS holds
// either form to seven workgroups, 364 against 275 us (630); one lane per pixel has no records in LDS.
// (tap sums per group instead of per channel, see backward_kernel's GV)
constexpr bool run_sums(int lpp, int reduce, int gv) { return gv < 4 && (lpp != 2 || reduce != 0); }
// The minimum of 8 channels: the third wave spills 28 bytes, two do not (one view, 173 x 194 x 91, 97 -> 87 us; two
// views, 40 x 60 x 30, four images, 29 -> 25.5); the mean is faster with it (two views, 136 against 148).
constexpr bool slim_double(int lpp, int corr, int reduce) { return corr == 2 && lpp > (reduce == 0 ? 1 : 2) && lpp <= 8; }
constexpr bool lean_backward(int nv, int lpp, int corr, int reduce, bool wide = false,
                             bool wide_real = false, int gv = 4) {
  return wide_real ||
         (nv == 1 && !wide &&
          (lpp == 16 || (lpp == 8 && corr != 1) ||
           (lpp == 4 && corr <= 4) || (lpp == 2 && (corr == 0 || (corr == 1 && reduce == 0))) ||
           (corr == 1 && run_sums(lpp, reduce, gv) && lpp >= 4)));
}
constexpr bool four_row_pairs(int corr, bool wide_real) { return corr == 3 || (corr == 5 && wide_real); }
// 32 channels: the gradients that have kernels for either window (six rows and eight).
constexpr bool two_windows(int corr, int reduce) { return (corr == 0 && reduce == 0) || corr == 2 || corr == 4; }
constexpr int backward_waves(int nv, int lpp, int corr = 0, int reduce = 1, bool wide = false,
                             bool wide_real = false, int gv = 4) {
  return wide_real ? (slim_double(lpp, corr, reduce) ? 3 : 2) : (lpp == 16 || corr == 5) && nv == 1               ? 3
         : lean_backward(nv, lpp, corr, reduce, wide, false, gv) ? 4
         : nv == 1 && lpp <= 8                       ? 3
         : nv <= 2                                   ? 2
                                                     : 1;
}

// REDUCE: 0 gradient of the mean (mask = number of accepted views), 1 gradient of the
// per-channel minimum / per-group maximum (mask = winning view per channel or group; a
// voxel is skipped when its first entry is negative, cost_volume_kernels_gpu.cu.cc:483-486)
// and of the summed-squared-difference minimum (mask = the voxel's winning view).
// DG: false when the caller does not want the depth gradient (a NULL output): the four
// depth-derivative weights per record and the 20 instructions per wave-iteration that use
// them drop out.
// PV: the depth hypotheses come from a per-voxel depth_grid (and the depth gradient is per
// voxel); a compile-time flag, because the kernel without the unused variant's code is
// measurably faster than one that tests a.depth_grid at run time.
// VLOOP: the workgroup's view group holds several views, which take turns (g.vper of them).
// A compile-time flag: the loop around the kernel's body costs the wide instantiations
// registers they do not have (the 32-channel kernel spills with it).
// EIGHT: 32 channels with a window of eight rows, for many views.  kEightWide: 8 x 8 texels and the kernel
// without the slimming of lean_backward, three waves per SIMD (also the small launches' form of the minimum,
// any width); kEightTall: 8 x 6 over tiles of 4 x 2
// pixels, the slimmed form turned by ninety degrees.  The launcher decides (tiled_launch.inc).
// PAD: fewer channels than the pixel's lanes hold (20, 24, 28 on eight lanes).  The lanes past the
// last channel compute what the last lane computes and contribute nothing: their gradients are
// selected to zero (not multiplied: infinities), their window slots stay zero.  A quarter of the
// arithmetic is idle at 24 channels, but eight pixels share a wave and a scatter window where the
// lane-per-channel kernels have two pixels and none (training
// passes of 24 channels: minimum over five views, 63 x 85 x 37, 219 -> 110 us; warped features, 212 x
// 213 x 86, 627 -> 344 us).
// GV (CORR 1): group values per lane -- four (groups of one channel), two, or one (of four; a group of eight
// is one that two lanes share).  A compile-time flag: a run-time width in the depth loop cost the 8-channel
// kernels 5 % (bf16, four views, 512 x 640 x 8, two images: 373 -> 353 us).
// With fewer values than channels (kRunSums) everything a depth adds factors into its group value and the
// channels, which stay what they are while a run lasts: the tap sums are kept per group, sum of cost_grad *
// weight, and meet the reference channels when the run ends (in the window's addition), the taps there too
// (ref_grad); the depth gradient takes the taps against the reference, formed once per run (`proj`).  Per
// depth 10 operations per group where the channel loop takes 15 per channel, and 16 to 28 registers less,
// which with 32 channels are a fourth wave per SIMD.  Gradient, two views unless said, 128 x 160: 32 channels in 8
// groups x 48 104 -> 90 us (maximum, three views, 241 -> 179), in 4 groups, six views, x 64 378 -> 334; 64
// channels in groups of four, maximum, 178 -> 154; 16 channels in 8 groups, maximum, four views, 150 x 200 x
// 32, 241 -> 185; double 139 -> 130; 8 channels, maximum, bf16 as above, 609 -> 428.  The mean of 8 channels
// keeps the channel loop: with 32 pixels in a wave a run ends at nearly every depth, and what a run costs
// more is what its depths save (537 -> 545 us for the training pass with bf16 run sums).  Errors against
// 64-bit sums are the channel loop's or below (1.03e-7 and 1.02e-7 of the norm; it: 1.04e-7, 1.05e-7).
template <typename S, int VEC, int LPP, int NV, int CORR, int REDUCE = 0, bool DG = true,
          bool PV = (CORR == 1), bool VLOOP = false, int EIGHT = kNotEight, bool PAD = false, int GV = 4>
__global__ __launch_bounds__(64, backward_waves(NV, LPP, CORR, REDUCE, EIGHT == kEightWide, sizeof(S) == 8, GV)) void backward_kernel(
    const Args<S> a, const Geometry g) {
  using R = typename Storage<S>::Real;
  using R4 = Four<R>;
  constexpr bool kDouble = sizeof(S) == 8;
  constexpr int GAP = lane_gap(LPP, CORR, (int)sizeof(S), PAD);
  constexpr bool kLean = lean_backward(NV, LPP, CORR, REDUCE, EIGHT == kEightWide, kDouble, GV);
  constexpr bool kSlim = kDouble && slim_double(LPP, CORR, REDUCE);
  constexpr int kForm = !(kLean && LPP == 8)                       ? kPlainWindow
                        : kSlim || four_row_pairs(CORR, kDouble) ? kFourRows
                        : EIGHT == kEightTall                      ? kSixColumns
                                                                   : kSixRows;
  using WN = Window<VEC, LPP, kForm>;
  constexpr int PPW = 64 / LPP;
  constexpr bool kWide = sizeof(S) == 2;  // gradients accumulate in fp32 images
  extern __shared__ __align__(16) unsigned char smem[];
  Tile<LPP> t;
  if (!locate_tile<S, LPP, EIGHT == kEightTall>(a, g, t)) return;
  const int C = PAD ? (int)a.C : VEC * LPP;
  constexpr int kUnit = cell_unit(VEC * LPP, PAD);
  const int D = (int)a.D, N = (int)a.N, srcH = (int)a.srcH, srcW = (int)a.srcW;
  const R half = a.half;
  constexpr bool per_voxel_depth = PV;
  constexpr bool kDstWords = !kSlim || PV;
  // byte offsets of the record arrays; a record is addressed as (lane-dependent byte offset)
  // + (compile-time constant), so that the constant lands in the instruction's offset field
  constexpr int kB = (int)sizeof(R), kB4 = (int)sizeof(R4);
  constexpr int kWts = 0, kDwt = kWts + (kSlim ? 0 : NV * 64 * kB4), kCell = kDwt + NV * 64 * kB4,
                kOff = kCell + NV * 64 * 8, kScl = kOff + NV * 64 * 4, kDst = kScl + 64 * kB;
  const unsigned p4 = (unsigned)t.p * 4u;                      // reader: pixel p
  const unsigned q4 = (unsigned)(t.cl * PPW + t.p) * 4u;       // writer: lane (p, j)
  const unsigned p1 = p4 * (unsigned)(kB / 4), q1 = q4 * (unsigned)(kB / 4);  // one R per voxel
  const unsigned pw = p4 * (unsigned)kB, qw = q4 * (unsigned)kB;               // four
  int *s_list = NV == 1 ? reinterpret_cast<int *>(smem)
                        : reinterpret_cast<int *>(smem + (LPP > 1 ? kDst + 64 * kB : 0));
  R *s_data = reinterpret_cast<R *>(smem + backward_record_bytes<R, VEC, LPP, NV, kForm, kSlim, kDstWords>());
  R *s_stage = s_data + NV * WN::SLOTS * WN::STRIDE;
  int *s_tags = reinterpret_cast<int *>(s_stage + 4 * WN::C);  // narrow pixels: claim words
  static_assert(LPP > kClaimLanes || NV == 1, "one set of claim words: one view per workgroup");
  int *s_own_list = s_tags + (LPP <= kClaimLanes ? WN::SLOTS : 0);
  // (LPP == 1: the records are in registers)
  int *s_move_list = LPP == 1                                         ? s_list
                     : backward_list_bytes<R, VEC, LPP, kForm>() > 0 ? s_own_list
                                                                 : reinterpret_cast<int *>(s_stage);
  // The source gradient of a channel is an outer product, four weights times one gradient per depth: for
  // the warp alone, with four lanes and more per pixel, the matrix cores add it, a block of four
  // lanes (channels) at a time and the lanes' channels one after the other: four instructions instead of
  // sixteen multiply-adds, in the same single rounding.  They write every lane, whatever the execution
  // mask: a lane without a sample takes part with a gradient of zero.  (Samples of 16 channels, three views, 97 x 129 x 40, two images: 103 -> 98 us at
  // four waves per SIMD, 94-96 with the matrix cores; 32 channels, five views, 247 x 274 x 72: 1945 ->
  // 1850 us; its error against 64-bit sums is that of the multiply-adds.)  The other gradients
  // have no registers left for it: 32 channels, two views, spill 32-52 bytes at four waves and lose
  // more (252 -> 263-338 us), 16 channels and CostAggregate gain nothing.
  constexpr bool kMatrix = CORR == 4 && !kDouble && LPP >= 4;
  using Sums = typename std::conditional<kMatrix, f32x4, LooseSums<R>>::type;
  const unsigned own_tap = pw + (unsigned)(t.lane & 3) * (unsigned)kB;
  // CORR 3 only: reference rows, sample rows
  R *s_v3 = reinterpret_cast<R *>(s_own_list + backward_list_bytes<R, VEC, LPP, kForm>() / 4);
  static_assert(!best_pair_op(CORR) || (NV == 1 && LPP > 1 && VEC == 4), "CostVolumeV3: one view, wide pixels");
  const R base = per_voxel_depth ? R(0) : a.base_plane[t.pix];
  static_assert(!PAD || !best_pair_op(CORR), "CostVolumeV3: whole pixels");
  const int cm = PAD ? C : WN::C;
  const bool ch_ok = !PAD || t.cl * VEC < C;
  const int clc = PAD ? min(t.cl, C / VEC - 1) : t.cl;  // the lane whose channels this lane reads
  const int ch0 = lane_first(clc, GAP);
  R ref[VEC];
  if constexpr (CORR != 4) {
    load_vec<S, VEC, false, GAP>(a.ref + t.pix * C + ch0, ref);
    if constexpr (best_pair_op(CORR)) {
#pragma unroll
      for (int c = 0; c < VEC; ++c) s_v3[t.p * (VEC * LPP) + t.cl * VEC + c] = ref[c];
    }
  } else {
    static_assert(CORR != 4 || NV == 1, "the warp-only gradient runs one view per workgroup");
#pragma unroll
    for (int c = 0; c < VEC; ++c) ref[c] = R(0);
  }
  if constexpr (PAD && run_sums(LPP, REDUCE, GV)) {  // (idle lanes: their window slots stay zero)
#pragma unroll
    for (int c = 0; c < VEC; ++c) ref[c] = ch_ok ? ref[c] : R(0);
  }
  constexpr int kWideSub = CORR == 5 ? 2 : 8;  // CostVolumeV3: the wider of the kernel's two group widths
  Two<R> ends{};
  if constexpr (CORR == 5 && REDUCE == 0) ends = ref_ends<LPP>(ref);
  const int64_t view_elems = (int64_t)srcH * srcW * C;
  R *src_grad_img;
  if constexpr (kWide) src_grad_img = a.src_grad_acc;
  else src_grad_img = a.src_grad;
  const int row_step = srcW * C;
  const unsigned lane_ch = (unsigned)ch0;
  R racc[VEC];
#pragma unroll
  for (int c = 0; c < VEC; ++c) racc[c] = R(0);
  R dacc = R(0);  // base-plane gradient partial of this lane

  // CORR: 0 squared difference per channel, 1 group correlation, 2 squared difference
  // summed over all channels (one upstream gradient per voxel), 4 the warp alone: one
  // upstream-gradient row and one 0/1 mask entry per (voxel, view)
  // (feature_aggregate_kernels_gpu.cu.cc:219-326)
  // 3: CostVolumeV3, one upstream gradient per voxel that flows through the best group pair
  constexpr bool kVoxelGrad = CORR == 2 || best_pair_op(CORR);
  // One winning view per voxel (or group): a view's runs are few and end far apart in depth.  An open
  // run from a cell left long ago need not make a chunk spread (kEndLeft), and where few runs end at
  // a depth moving the window to them costs more than adding them to memory (kFewRuns, in pixels of
  // the wave; end_spread_runs).  Four views, 136 x 176, 24 planes from 0.9: best pair of 32 channels
  // 276 -> 186 us (189 with every run outside the window added to memory), dense planes 378 -> 341 us;
  // CostAggregate of 16 and 8 channels 144 -> 112 and 108 -> 71 us.  The lines: an eighth of the
  // pixels, but four for the best pair, whose gradient is bound by instructions and leaves the
  // atomics room (64 channels: none 407, two 313, four 273 us).  The gradients of CostAggregate with
  // 32 channels and more keep the runs left behind open: the check costs them more than it saves (two
  // views, dense: 181 us without, 187 with it).  Where a mean or every channel's own winner keeps
  // all runs short, most pixels of a tile end together and the window pays.
  constexpr bool kWinners = REDUCE == 1 && (kVoxelGrad || CORR == 1);
  constexpr bool kEndLeft = kWinners && (CORR != 2 || LPP < 8);
  constexpr int kFewRuns = !kWinners ? 0 : best_pair_op(CORR) ? 4 : PPW / 8;
  const int OC = CORR == 1 ? a.groups : kVoxelGrad ? 1 : C;
  static_assert(VEC == 4 && (GV == 4 || (CORR == 1 && (GV == 2 || GV == 1))), "group values per lane");
  constexpr bool kRunSums = run_sums(LPP, REDUCE, GV);
  constexpr int NS = kRunSums ? GV : VEC;  // sums per tap
  const int goff = CORR == 1 ? group_offset<VEC>(clc, g.sub) : ch0;
  const int d_lo = t.d_lo, d_hi = t.d_hi;
  // upstream-gradient rows fetched ahead; the MIN reduce stages the mask rows beside them
  constexpr int PFMAX = (REDUCE || kLean) ? 4 : 8;
  constexpr int PF = LPP < PFMAX ? LPP : PFMAX;
  constexpr bool kMaskRows = REDUCE == 1 && !kVoxelGrad;
  static_assert(!kMaskRows || NV == 1, "the MIN gradient runs one view per workgroup");
  constexpr bool kWonMasks = kMaskRows && kLean && !kDouble && LPP <= 8;  // (find_won)
  // mask entries per voxel: the MIN reduce of CostVolumeV3 records (view, reference group,
  // source group)
  const int mask_w = kMaskRows ? OC : (best_pair_op(CORR) && REDUCE == 1) ? 3 : 1;
  // element steps from one depth to the next in the upstream gradient and in the mask
  const int cg_step = CORR == 4 ? N * C : OC;
  const int cnt_step = CORR == 4 ? N : mask_w;
  const R *dv_src = per_voxel_depth ? a.depth_grid + t.pix * D : a.offsets + (int64_t)t.b * D;
  // The views of this workgroup's group take turns (NV at a time; NV = 1 in every launch):
  // each gets the scatter window to itself and leaves it empty.  What belongs to the pixel
  // (reference gradient, depth gradients, the upstream rows in the caches) is shared, so a
  // group of all N views needs no atomics for the pixel-owned outputs.
  const int first_view = t.view0;
  const int group_views = VLOOP ? min(g.vper > NV ? g.vper : NV, N - first_view) : NV;
  for (int vi = 0; vi < group_views; vi += NV) {
  t.view0 = first_view + vi;
  if constexpr (VLOOP) {
    // The lane index as a value the compiler cannot see through: without this it computes
    // everything that depends only on the lane (slot and row arithmetic of the window moves
    // and flushes) once in front of the view loop and keeps it in registers through all
    // views -- two dozen registers the depth loop needs.
    asm volatile("" : "+v"(t.lane), "+v"(t.cl), "+v"(t.p), "+v"(t.pix), "+v"(t.h), "+v"(t.w));
  }
  for (int k = t.lane * 4; k < NV * WN::SLOTS * WN::STRIDE; k += 256)
    *reinterpret_cast<R4 *>(s_data + k) = R4{R(0), R(0), R(0), R(0)};
  if constexpr (tagged_slots(LPP))
    for (int k = t.lane; k < WN::SLOTS; k += 64) s_tags[k] = -1;
  Cameras<NV, R> cam;
  if constexpr (!kSlim)
    load_cameras<S, NV>(a, t.b, t.view0, static_cast<R>(t.w) + half, static_cast<R>(t.h) + half, cam);
  int cam_w = t.w, cam_h = t.h;
  const S *view[NV];
  R *gview[NV];  // gradient image of the view, no lane offset
  int oy[NV], ox[NV];
#pragma unroll
  for (int n = 0; n < NV; ++n) {
    const int64_t vo = ((int64_t)t.b * N + (t.view0 + n < N ? t.view0 + n : 0)) * view_elems;
    view[n] = a.src + vo;  // uniform: taps are addressed as base + 32-bit lane offset
    gview[n] = src_grad_img + vo;
    oy[n] = ox[n] = WN::kNone;
  }
  constexpr bool kRaw = is_half<S>();
  Taps<S, VEC, kRaw> tap[NV];
  Sums sg[NV][NS];
  R proj[NV][4][kRunSums && DG ? GV : 1];  // kRunSums: the taps of the open run against the reference, per group
  int cur[NV];     // tap offset of the open run, -1: none
  int2 cell[NV];   // its slots and key (bit 31: inside the window)
  unsigned ring_rows[NV];  // (without tags) ring rows of the window this lane's accepted cells mapped to
#pragma unroll
  for (int n = 0; n < NV; ++n) {
    cur[n] = -1;
    ring_rows[n] = 0u;
    cell[n] = make_int2(0, 0);
#pragma unroll
    for (int c = 0; c < NS; ++c) sg[n][c] = Sums{R(0), R(0), R(0), R(0)};
  }
  // kRunSums: the reference gradient of a run that ends (its taps are still at hand)
  auto take_run = [&](int n) __attribute__((always_inline)) {
    if constexpr (kRunSums) {
#pragma unroll
      for (int c = 0; c < VEC; ++c) {
        R run = kRaw ? mad(tap[n](0, c), sg[n][c * NS / VEC][0], R(0)) : tap[n](0, c) * sg[n][c * NS / VEC][0];  // (summed by itself: one rounding per run in racc)
#pragma unroll
        for (int k = 1; k < 4; ++k) run = mad(tap[n](k, c), sg[n][c * NS / VEC][k], run);
        racc[c] += run;
      }
    }
  };
  const S *cg_lane =
      CORR == 4 ? a.cost_grad + (t.pix * D * N + t.view0) * C + ch0
                : a.cost_grad + t.pix * D * OC + (kVoxelGrad ? 0 : goff);
  const int32_t *cnt_src = CORR == 4 ? a.mask_in + t.pix * D * N + t.view0
                                     : a.mask_in + t.pix * D * mask_w;
  const int32_t *mask_lane = cnt_src + goff;  // this lane's part of a mask row
  // the pixel's depth gradients: the first view of a group that holds them all stores, the
  // later ones add (same lane, same address); several groups add atomically
  const bool dg_store = g.ngroups == 1 && vi == 0, dg_own = g.ngroups == 1;
  // Runs of a spread chunk that end now (`fire`: whole pixels; called by all lanes).  The
  // samples of such a chunk land so far apart (hypotheses close to the cameras, wide baselines,
  // few planes far apart) that its cells do not fit the window together, but the runs that end
  // at one depth lie about as close to each other as the tile's pixels do, so the window moves
  // to them: neighbouring pixels share most of their texels (2 x 4 pixels: about 15 instead of
  // 32 taps), which then leave as one dense run of atomics each, and the rate of the atomics is
  // what bounds such a launch (32 channels, six views, depths from 0.5, 15-degree rotations:
  // 18.5 -> 13.3 ms against every cell of such a chunk adding its four texels to memory by itself;
  // minimum over two views, 260 x 372, twelve planes from 1.7 to 16: 632 -> 351 us).  A cell that is
  // still outside (pixels of one depth further apart than the window, on strongly magnified views)
  // goes to memory by itself, and so do a few runs of seldom winners (kFewRuns).  CostVolumeV3's
  // gradient of a mean spends its time on the pair search: 24 far-apart planes of 32 channels 0-3 %
  // slower than with every cell added to memory, of 16 channels 1.2-1.5x faster; dense planes 0.8 %
  // slower (188.4 -> 189.9 us) for the block in its loop.
  auto end_spread_runs = [&](int n, bool fire) __attribute__((always_inline)) {
    // (the lane index as a value the compiler cannot see through: what the window's functions
    // derive from it would be computed in front of all chunks and held through the depth loop)
    int lane = t.lane;
    if constexpr (LPP < 8) asm volatile("" : "+v"(lane));
    const int cl = LPP < 8 ? lane % LPP : t.cl;
    const int key = cell[n].y & 0x7fffffff;
    bool in = WN::inside(key, oy[n], ox[n]);
    const unsigned long long outside = __ballot(fire && !in);
    if (outside != 0ull) {
      if (kFewRuns == 0 || __popcll(outside) > kFewRuns * LPP) {
        const Box b = wave_box(fire ? key : kNoLow, fire ? key : kNoHigh);
        const int sy = WN::ROWS - (b.y1 - b.y0 + 1), sx = WN::COLS - (b.x1 - b.x0 + 1);
        window_move<VEC, LPP, kForm, 2>(oy[n], ox[n], b.y0 - (sy > 0 ? sy / 2 : 0), b.x0 - (sx > 0 ? sx / 2 : 0),
                                    s_data + n * WN::SLOTS * WN::STRIDE, s_tags, s_move_list, gview[n], srcW, lane, cm);
        in = WN::inside(key, oy[n], ox[n]);
      }
      const bool out = fire && !in;
      const unsigned long long m = __ballot(out);
      if (m != 0ull) {
        if (out) take_run(n);
        flush_cells_to_memory<VEC, LPP, GAP>(m, out, key, sg[n], ref, s_stage, gview[n], srcW, lane, cl, cm);
        if (out) cur[n] = -1;
      }
    }
    if (fire) cell[n].y = in ? (key | WN::kInside) : key;
  };
  wave_sync();
  for (int d0 = d_lo; d0 < d_hi; d0 += LPP) {
    // Depth hypothesis and valid-view count of lane (p, j)'s voxel: requested before the
    // chunk's upstream-gradient rows, because loads return in order and the reprojection
    // should wait for these two words only.
    R dv = R(1), cg_vox = R(0);
    int cnt = REDUCE ? -1 : 0;  // "nothing to do" for a lane without a voxel
    int v3_pair = kNoPair;
    if (d0 + t.cl < d_hi) {
      dv = dv_src[d0 + t.cl];
      if (t.pix_ok) cnt = cnt_src[(int64_t)(d0 + t.cl) * cnt_step];
      if constexpr (kVoxelGrad)  // the voxel's one upstream gradient rides with its record
        cg_vox = reinterpret_cast<const R *>(cg_lane)[d0 + t.cl];
      if constexpr (best_pair_op(CORR) && REDUCE == 1) {
        if (t.pix_ok) {
          const int64_t m3 = (int64_t)(d0 + t.cl) * 3;
          const int gi = cnt_src[m3 + 1], gs = cnt_src[m3 + 2];
          // a recorded group outside the image's groups: the voxel is skipped
          if ((unsigned)gi < (unsigned)a.groups && (unsigned)gs < (unsigned)a.groups)
            v3_pair = gs * kPairRow + gi;
          else
            cnt = -1;
        }
      }
    }
    int r_off[NV];
    int2 r_cell[NV];
    R r_scl = R(0);
    R4 r_wts[NV], r_dwt[NV];
    bool spread[NV];  // the cells of this chunk and the open ones do not fit the window together
    // Issue the loads of this chunk's cost_grad rows now, unconditionally, so that the
    // reprojection below overlaps their latency.  Through the caches: the workgroups of a
    // tile's views read the same rows (streamed, only about a third of the later reads found
    // them in L2).  At three waves per SIMD that was worth 2 % and cost the next forward launch
    // 5 us; at four waves it is worth 4 %, the forward launch does not notice, and 13 % less
    // is fetched.  One cache state is slower this way (by 4 %): every line dirty with another
    // kernel's output, which a load that allocates has to push out first.
    // (whole rows are kept as loaded and widened to float where a depth uses them; group
    // rows are widened here and kept as float bits)
    RawWord<S> cgw[kVoxelGrad ? 1 : PF][(CORR == 0 || CORR == 4) ? raw_words<S, VEC>() : GV];
    int mrow[kMaskRows ? PF : 1][GV];
    auto load_rows = [&](int first) {
      if constexpr (kMaskRows) {
#pragma unroll
        for (int jj = 0; jj < PF; ++jj) {
          const int d = min(first + jj, d_hi - 1);
          const int32_t *m = mask_lane + (int64_t)d * OC;
          if constexpr (GAP != 2) {
            const int2 lo = *reinterpret_cast<const int2 *>(m), hi = *reinterpret_cast<const int2 *>(m + GAP);
            mrow[jj][0] = lo.x, mrow[jj][1] = lo.y, mrow[jj][2] = hi.x, mrow[jj][3] = hi.y;
          } else if constexpr (GV == 4) {
            typedef int i32x4 __attribute__((ext_vector_type(4)));
            const i32x4 v = *reinterpret_cast<const i32x4 *>(m);
            mrow[jj][0] = v[0], mrow[jj][1] = v[1], mrow[jj][2] = v[2], mrow[jj][3] = v[3];
          } else if constexpr (GV == 2) {
            typedef int i32x2 __attribute__((ext_vector_type(2)));
            const i32x2 v = *reinterpret_cast<const i32x2 *>(m);
            mrow[jj][0] = v[0], mrow[jj][1] = v[1];
          } else {
            mrow[jj][0] = *m;
          }
        }
      }
      if constexpr (CORR == 1) {
#pragma unroll
        for (int jj = 0; jj < PF; ++jj) {
          const int d = min(first + jj, d_hi - 1);
          load_vec<S, GV, false>(cg_lane + (int64_t)d * cg_step, reinterpret_cast<R *>(cgw[jj]));
        }
      }
#pragma unroll
      for (int jj = 0; jj < PF; ++jj) {
        const int d = min(first + jj, d_hi - 1);
        const S *src_cg = cg_lane + (int64_t)d * cg_step;
        // (each view of FeatureAggregate has rows of its own: streamed where they cover whole
        // lines)
        if constexpr (CORR == 0)
          load_raw<S, VEC, false, GAP>(src_cg, cgw[jj]);
        if constexpr (CORR == 4)
          load_raw<S, VEC, whole_lines(VEC * LPP, (int)sizeof(S)), GAP>(src_cg, cgw[jj]);
      }
    };
    // Only the channels (groups) this view won contribute: the rest of a staged row becomes zero.  The
    // comparisons are made when the winners arrive, whose first entry the reprojection waits for anyway, and
    // kept as lane masks in scalar registers, so that the winners hold no registers through the walk.
    unsigned long long won[kWonMasks ? PF : 1][GV];
    auto find_won = [&]() __attribute__((always_inline)) {
      if constexpr (kWonMasks) {
#pragma unroll
        for (int jj = 0; jj < PF; ++jj)
#pragma unroll
          for (int i = 0; i < GV; ++i) won[jj][i] = __ballot(mrow[jj][i] == t.view0);
      }
    };
    auto keep_won = [&]() __attribute__((always_inline)) {
      if constexpr (kWonMasks) {
        auto select = [](uint32_t w, unsigned long long m) __attribute__((always_inline)) {
          return __builtin_amdgcn_inverse_ballot_w64(m) ? w : 0u;
        };
#pragma unroll
        for (int jj = 0; jj < PF; ++jj) {
          if constexpr (sizeof(S) == 2 && CORR == 0) {  // (two channels per word)
#pragma unroll
            for (int i = 0; i < GV / 2; ++i)
              cgw[jj][i] &= select(0xffffu, won[jj][2 * i]) | select(0xffff0000u, won[jj][2 * i + 1]);
          } else {
#pragma unroll
            for (int i = 0; i < GV; ++i) cgw[jj][i] = select(cgw[jj][i], won[jj][i]);
          }
        }
      }
    };
    if constexpr (!kVoxelGrad) load_rows(d0);
    find_won();
    {
      const R depth = d0 + t.cl < d_hi ? (per_voxel_depth ? dv : base + dv) : R(1);
      // factor the reduce applies to the upstream gradient: squared difference 2/k,
      // correlation 1/k, summed squared difference 2*cost_grad/(k*C) (the whole per-voxel
      // factor); zero marks a voxel that contributes nothing
      // (a division in double is fifty instructions: there the reciprocal serves)
      if constexpr (kSlim) {
        // (computed again for every chunk: as values of the whole walk they would be 24 registers; the
        // compiler would make them that if it could see through the pixel's coordinates)
        asm volatile("" : "+v"(cam_w), "+v"(cam_h));
        load_cameras<S, NV>(a, t.b, t.view0, static_cast<R>(cam_w) + half, static_cast<R>(cam_h) + half, cam);
      }
      static_assert(NV == 1, "one view at a time");
      bool nothing = false;
      R scl = R(0);
      if constexpr (REDUCE == 0) {
        if (cnt > 0) {
          if constexpr (CORR == 2 && kDouble)
            scl = R(2) * cg_vox * quick_recip(static_cast<R>(cnt * C));
          else if constexpr (CORR == 2)
            scl = R(2) * (cg_vox / static_cast<R>(cnt * C));
          else if constexpr (best_pair_op(CORR))
            scl = cg_vox / static_cast<R>(cnt);  // cost_volume_kernels_gpu_v3.cu.cc:426
          else
            scl = (CORR == 0 ? R(2) : R(1)) * quick_recip(static_cast<R>(cnt));
        }
      } else {
        // no division by the view count; `cnt` holds the first mask entry of the voxel (or,
        // for the summed squared difference, its winning view)
        if constexpr (CORR == 2) {
          if (cnt == t.view0) scl = R(2) * (cg_vox / static_cast<R>(C));
        } else if constexpr (best_pair_op(CORR)) {
          if (cnt == t.view0) scl = cg_vox;  // cost_volume_kernels_gpu_v3.cu.cc:621-622
        } else {
          if (cnt >= 0) scl = CORR == 0 ? R(2) : R(1);
        }
      }
#pragma unroll
      for (int n = 0; n < NV; ++n) {
        // A chunk without a voxel that counts -- outside this view, or, where every voxel has one winner, won by
        // the others -- leaves everything as it is.  (Not where every voxel's depth gradient is stored.)
        if (!PV && kWinners && __ballot(scl != R(0)) == 0ull) {
          nothing = true;
          break;
        }
        Hit<R> hit;
        reproject<NV, R>(cam, n, depth, half, g.src_h_max, g.src_w_max, srcW, t.view0 + n < N && scl != R(0), hit);
        if (!PV && __ballot(hit.cell >= 0) == 0ull) {
          nothing = true;
          break;
        }
        R4 dw4 = R4{R(0), R(0), R(0), R(0)};
        if constexpr (DG) {
          // d(sample)/d(depth) = sum over taps of dwt * tap, from
          //   d/d(src_h) = t1*dw + (t10 - t00),  d/d(src_w) = t1*dh + (t01 - t00),
          //   t1 = t11 - t10 - t01 + t00, chained through the perspective divide.
          const R inv = quick_recip(hit.z * hit.z);
          const R ah = (cam.hc[n] * hit.z - cam.zc[n] * hit.h3d) * inv;
          const R aw = (cam.wc[n] * hit.z - cam.zc[n] * hit.w3d) * inv;
          const R cp = ah * hit.dw + aw * hit.dh;
          dw4 = R4{cp - ah - aw, aw - cp, cp, ah - cp};
          if constexpr (kSlim) dw4 = R4{R(0), R(0), ah, aw};  // taps 00, 01, 11, 10
        }
        // The scatter window has to cover this chunk's cells and the cell still open from
        // the last chunk.  Usually it already does (one vote); otherwise it is centred on
        // their bounding box.  A box larger than the window: the window follows the runs that
        // end, depth by depth (end_spread_runs).
        const bool valid = hit.cell >= 0;
        if constexpr (kMatrix) {  // (the matrix cores multiply the weights of lanes without a sample too, by zero)
          if (!valid) hit.k00 = hit.k01 = hit.k11 = hit.k10 = R(0);
        }
        const int r0 = WN::ring_row((unsigned)hit.key >> 16 & 0x7fffu), r1 = WN::template ring_next<WN::ROWS>(r0);
        if constexpr (!tagged_slots(LPP))
          if (valid) ring_rows[n] |= (1u << r0) | (1u << r1);
        bool in_new = !valid || WN::inside(hit.key, oy[n], ox[n]);
        spread[n] = false;
        if (__ballot(!(in_new && (cur[n] < 0 || cell[n].y < 0))) != 0ull) {
          int lo = valid ? hit.key : kNoLow, hi = valid ? hit.key : kNoHigh;
          if (cur[n] >= 0) {
            const int open = cell[n].y & 0x7fffffff;
            lo = min_halves(lo, open), hi = max_halves(hi, open);
          }
          Box b = wave_box(lo, hi);
          int sy = WN::ROWS - (b.y1 - b.y0 + 1), sx = WN::COLS - (b.x1 - b.x0 + 1);  // slack
          spread[n] = sy < 0 || sx < 0;
          if constexpr (kEndLeft) {
            if (spread[n] && __ballot(valid) != 0ull) {
              // without the open runs: where the chunk's cells fit, the runs it leaves behind end
              b = wave_box(valid ? hit.key : kNoLow, valid ? hit.key : kNoHigh);
              sy = WN::ROWS - (b.y1 - b.y0 + 1), sx = WN::COLS - (b.x1 - b.x0 + 1);
              spread[n] = sy < 0 || sx < 0;
              const int key = cell[n].y & 0x7fffffff;
              const bool left = !spread[n] && cur[n] >= 0 && !WN::inside(key, b.y0 - sy / 2, b.x0 - sx / 2);
              const unsigned long long m = __ballot(left);
              if (m != 0ull) {
                if (left) take_run(n);
                flush_cells_to_memory<VEC, LPP, GAP>(m, left, key, sg[n], ref, s_stage, gview[n], srcW, t.lane, t.cl, cm);
                if (left) cur[n] = -1;
              }
            }
          }
          if (spread[n]) {
            in_new = false;  // decided when the run ends
            cell[n].y &= 0x7fffffff;
          } else {
            window_move<VEC, LPP, kForm>(oy[n], ox[n], b.y0 - sy / 2, b.x0 - sx / 2,
                                  s_data + n * WN::SLOTS * WN::STRIDE, s_tags, s_list, gview[n], srcW, t.lane, cm);
            in_new = true;
            cell[n].y |= WN::kInside;
          }
        }
        const int2 rec = make_int2(WN::kPacked ? (int)WN::pack_slots(r0, r1, (unsigned)hit.key & 0xffffu) : 0,
                                   (valid && in_new) ? (hit.key | WN::kInside) : hit.key);
        if constexpr (LPP > 1) {
          lds_at<int>(smem, q4, kOff + (n * LPP * PPW) * 4) = PAD && valid ? hit.cell * C : hit.cell;
          lds_at<int2>(smem, q4 * 2u, kCell + (n * LPP * PPW) * 8) = rec;
          if constexpr (kSlim) {
            lds_at<R4>(smem, qw, kWts + (n * LPP * PPW) * kB4) = R4{hit.dh, hit.dw, dw4.z, dw4.w};
          } else {
            lds_at<R4>(smem, qw, kWts + (n * LPP * PPW) * kB4) = R4{hit.k00, hit.k01, hit.k11, hit.k10};
            if constexpr (DG) lds_at<R4>(smem, qw, kDwt + (n * LPP * PPW) * kB4) = dw4;
          }
        } else {
          r_off[n] = hit.cell;
          r_cell[n] = rec;
          r_wts[n] = R4{hit.k00, hit.k01, hit.k11, hit.k10};
          r_dwt[n] = dw4;
        }
      }
      if (nothing) continue;
      if constexpr (LPP > 1) {
        lds_at<R>(smem, q1, kScl) = scl;
        if constexpr (best_pair_op(CORR))
          lds_at<int>(smem, q4, kDst) = v3_pair;  // (this op has no per-voxel depth gradient)
        else if constexpr (kDstWords)
          lds_at<R>(smem, q1, kDst) = R(0);
      } else {
        r_scl = scl;
      }
    }
    if constexpr (LPP > 1) wave_sync();
    keep_won();
    int rb_off[2][NV];
    R4 rb_wt[2][NV], rb_dwt[2][NV];
    R rb_scl[2], own_w = R(0);
#pragma unroll
    for (int n = 0; n < NV; ++n) {
      if constexpr (LPP > 1) {
        rb_off[0][n] = lds_at<int>(smem, p4, kOff + (n * LPP * PPW) * 4);
        rb_wt[0][n] = lds_at<R4>(smem, pw, kWts + (n * LPP * PPW) * kB4);
        if constexpr (DG && !kSlim)
          rb_dwt[0][n] = lds_at<R4>(smem, pw, kDwt + (n * LPP * PPW) * kB4);
        else
          rb_dwt[0][n] = R4{R(0), R(0), R(0), R(0)};
      } else {
        rb_off[0][n] = r_off[n];
        rb_wt[0][n] = r_wts[n];
        rb_dwt[0][n] = r_dwt[n];
      }
    }
    if constexpr (kMatrix) own_w = lds_at<R>(smem, own_tap, kWts);
    if constexpr (LPP > 1)
      rb_scl[0] = lds_at<R>(smem, p1, kScl);
    else
      rb_scl[0] = r_scl;
#pragma unroll
    for (int jj = 0; jj < LPP; ++jj) {
      const int d = d0 + jj;
      // (no early exit past d_hi: the records of such depths carry a zero factor and no tap
      // offset, the row loads are clamped, and a loop without exits compiles to faster code)
      if constexpr (LPP > PF && !kVoxelGrad) {
        if (jj > 0 && jj % PF == 0) {  // next part of a deep chunk
          load_rows(d0 + jj);
          find_won();
          keep_won();
        }
      }
      // The records of the NEXT depth are requested now, so that their LDS latency overlaps
      // this depth's arithmetic (jj is unrolled: the buffer index is a compile-time constant).
      // (a lean kernel reads the records of depth jj here, into the one set it keeps)
      const int cb = kLean ? 0 : (jj & 1), nb = kLean ? 0 : (cb ^ 1);
      constexpr int kAhead = kLean ? 0 : 1;
      if constexpr (LPP > 1) {
        if (kLean ? jj > 0 : jj + 1 < LPP) {
#pragma unroll
          for (int n = 0; n < NV; ++n) {
            rb_off[nb][n] = lds_at<int>(smem, p4, kOff + ((n * LPP + jj + kAhead) * PPW) * 4);
            rb_wt[nb][n] = lds_at<R4>(smem, pw, kWts + ((n * LPP + jj + kAhead) * PPW) * kB4);
            if constexpr (DG && !kSlim)
              rb_dwt[nb][n] = lds_at<R4>(smem, pw, kDwt + ((n * LPP + jj + kAhead) * PPW) * kB4);
            else
              rb_dwt[nb][n] = R4{R(0), R(0), R(0), R(0)};
          }
          rb_scl[nb] = lds_at<R>(smem, p1, kScl + ((jj + kAhead) * PPW) * kB);
        }
      }
      const int *rec_off = rb_off[cb];
      const R4 *rec_wt = rb_wt[cb], *rec_dwt = rb_dwt[cb];
      const R scl = rb_scl[cb];
      if constexpr (kMatrix)
        if (jj > 0) own_w = lds_at<R>(smem, own_tap, kWts + (jj * PPW) * kB4);
      R gmat[VEC];  // d(loss)/d(sample) of this lane's channels for the matrix cores
#pragma unroll
      for (int c = 0; c < VEC; ++c) gmat[c] = R(0);
      R dvox = R(0);  // this lane's share of d(loss)/d(depth of this voxel)
#pragma unroll
      for (int n = 0; n < NV; ++n) {
        if (spread[n]) {  // uniform, and false for the whole chunk in the usual case
          const bool fire = scl != R(0) && rec_off[n] >= 0 && rec_off[n] != cur[n] && cur[n] >= 0;
          end_spread_runs(n, fire);
        }
      }
      // (one view per workgroup: a tap offset implies a non-zero factor, phase 1 reprojects
      // only voxels that have one; one test instead of two per depth)
      if (NV == 1 ? rec_off[0] >= 0 : scl != R(0)) {
        R cg[GV];  // of this lane's channels (group correlation: groups)
        {
          R raw[GV];
          if constexpr (!kVoxelGrad) {
            if constexpr (CORR == 0 || CORR == 4)
              widen_raw<S, VEC>(cgw[jj % PF], raw);
            else
#pragma unroll
              for (int c = 0; c < GV; ++c) raw[c] = raw_to_real(cgw[jj % PF][c]);
          }
          if constexpr (kVoxelGrad) {
#pragma unroll
            for (int c = 0; c < GV; ++c) cg[c] = scl;
          } else if (CORR == 4) {
            // (each view of FeatureAggregate has rows of its own: no factor)
#pragma unroll
            for (int c = 0; c < GV; ++c) cg[c] = raw[c];
          } else {
#pragma unroll
            for (int c = 0; c < GV; ++c) cg[c] = kRaw && CORR == 0 ? mad(raw[c], scl, R(0)) : raw[c] * scl;
          }
          if constexpr (kMaskRows && !kWonMasks) {
            // only the channels (groups) this view won contribute
#pragma unroll
            for (int c = 0; c < GV; ++c)
              if (mrow[jj % PF][c] != t.view0) cg[c] = R(0);
          }
          if constexpr (PAD && kRunSums) {
#pragma unroll
            for (int c = 0; c < GV; ++c) cg[c] = ch_ok ? cg[c] : R(0);
          }
        }
#pragma unroll
        for (int n = 0; n < NV; ++n) {
          const int off = rec_off[n];
          R4 wt = rec_wt[n], dwt = rec_dwt[n];
          if constexpr (kSlim) {
            // (each weight the rounded product of its two factors, as reproject() has it: three of them
            // come cheaper by subtraction, and lose their relative accuracy where they are small)
            const R dh = wt.x, dw = wt.y, ah = wt.z, aw = wt.w, eh = R(1) - dh, ew = R(1) - dw;
            wt = R4{eh * ew, eh * dw, dh * dw, dh * ew};
            const R cp = mad(ah, dw, aw * dh), bp = aw - cp;
            dwt = R4{-ah - bp, bp, cp, ah - cp};
          }
          if (off >= 0) {
            if (off != cur[n]) {
              // (a run whose cell the window could not cover was closed by the uniform block
              // above, which left cur[n] = -1)
              // the run on the previous cell ends.  Start fetching the new cell's taps
              // first, then hand the old cell's image to the window while they arrive.
              if constexpr (kRunSums)
                if (cur[n] >= 0) take_run(n);
              load_cell<S, VEC, GAP, kUnit>(view[n], off, C, row_step, lane_ch, tap[n]);
              if (cur[n] >= 0)
                window_add<VEC, LPP, kLean, kForm, GAP>((unsigned)cell[n].x, cell[n].y, sg[n], ref,
                                            s_data + n * WN::SLOTS * WN::STRIDE, s_tags, t.lane, t.cl);
              cur[n] = off;
              if constexpr (LPP > 1)
                cell[n] = lds_at<int2>(smem, p4 * 2u, kCell + ((n * LPP + jj) * PPW) * 8);
              else
                cell[n] = r_cell[n];
              if constexpr (kRunSums && DG) {
#pragma unroll
                for (int k = 0; k < 4; ++k)
#pragma unroll
                  for (int i = 0; i < GV; ++i) {
                    constexpr int SUB = VEC / GV;
                    R sum = kRaw ? mad(ref[i * SUB], tap[n](k, i * SUB), R(0)) : ref[i * SUB] * tap[n](k, i * SUB);
#pragma unroll
                    for (int c = 1; c < SUB; ++c) sum = mad(ref[i * SUB + c], tap[n](k, i * SUB + c), sum);
                    proj[n][k][i] = sum;
                  }
              }
            }
            if constexpr (kRunSums) {
#pragma unroll
              for (int i = 0; i < GV; ++i) {
                sg[n][i][0] = mad(cg[i], wt.x, sg[n][i][0]);
                sg[n][i][1] = mad(cg[i], wt.y, sg[n][i][1]);
                sg[n][i][2] = mad(cg[i], wt.z, sg[n][i][2]);
                sg[n][i][3] = mad(cg[i], wt.w, sg[n][i][3]);
                if constexpr (DG) {
                  R ds = dwt.x * proj[n][0][i];
                  ds = mad(dwt.y, proj[n][1][i], ds);
                  ds = mad(dwt.z, proj[n][2][i], ds);
                  ds = mad(dwt.w, proj[n][3][i], ds);
                  dvox = mad(cg[i], ds, dvox);
                }
              }
            } else {
            R gs3[VEC];
            if constexpr (best_pair_op(CORR)) {
              const int pair = REDUCE ? lds_at<int>(smem, p4, kDst + (jj * PPW) * 4) : 0;
              if (g.sub == kWideSub)
                v3_pair_gradients<R, VEC, LPP, kWideSub, REDUCE>(wt, tap[n].v, ends, scl, pair, s_v3, t.p,
                                                                 t.cl, racc, gs3);
              else
                v3_pair_gradients<R, VEC, LPP, kWideSub / 2, REDUCE>(wt, tap[n].v, ends, scl, pair, s_v3, t.p,
                                                                     t.cl, racc, gs3);
            }
#pragma unroll
            for (int c = 0; c < VEC; ++c) {
              R gsrc;  // d(loss)/d(sample of this channel)
              if constexpr (best_pair_op(CORR)) {
                gsrc = gs3[c];
              } else if constexpr (CORR == 4) {
                gsrc = cg[c * GV / VEC];
              } else if (CORR != 1) {
                // (double: the sample first, then the difference: sums of the sample's parts are the
                // smaller numbers to round, and the lane-per-channel kernels have it so)
                R diff = kDouble ? wt.x * tap[n](0, c) : mad(wt.x, tap[n](0, c), -ref[c]);
                diff = mad(wt.y, tap[n](1, c), diff);
                diff = mad(wt.z, tap[n](2, c), diff);
                diff = mad(wt.w, tap[n](3, c), diff);
                if constexpr (kDouble) diff -= ref[c];
                gsrc = diff * cg[c * GV / VEC];
                racc[c] -= gsrc;
              } else {
                R smp = kRaw ? mad(wt.x, tap[n](0, c), R(0)) : wt.x * tap[n](0, c);
                smp = mad(wt.y, tap[n](1, c), smp);
                smp = mad(wt.z, tap[n](2, c), smp);
                smp = mad(wt.w, tap[n](3, c), smp);
                racc[c] = mad(cg[c * GV / VEC], smp, racc[c]);
                gsrc = cg[c * GV / VEC] * ref[c];
              }
              if constexpr (PAD) gsrc = ch_ok ? gsrc : R(0);
              if constexpr (kMatrix) {
                gmat[c] = gsrc;
              } else {
                sg[n][c][0] = mad(gsrc, wt.x, sg[n][c][0]);
                sg[n][c][1] = mad(gsrc, wt.y, sg[n][c][1]);
                sg[n][c][2] = mad(gsrc, wt.z, sg[n][c][2]);
                sg[n][c][3] = mad(gsrc, wt.w, sg[n][c][3]);
              }
              if constexpr (DG) {
                R ds = kRaw ? mad(dwt.x, tap[n](0, c), R(0)) : dwt.x * tap[n](0, c);
                ds = mad(dwt.y, tap[n](1, c), ds);
                ds = mad(dwt.z, tap[n](2, c), ds);
                ds = mad(dwt.w, tap[n](3, c), ds);
                dvox = mad(gsrc, ds, dvox);
              }
            }
            }
          }
        }
      }
      if constexpr (kMatrix) {
#pragma unroll
        for (int c = 0; c < VEC; ++c)
          sg[0][c] = __builtin_amdgcn_mfma_f32_4x4x1f32(own_w, gmat[c], sg[0][c], 0, 0, 0);
      }
      if constexpr (PAD && DG) dvox = ch_ok ? dvox : R(0);
      if constexpr (!DG) {
        // no depth gradient wanted
      } else if (per_voxel_depth) {
        if constexpr (LPP > 1) {
          const R tot = group_sum<LPP>(dvox);
          if (t.cl == 0) lds_at<R>(smem, p1, kDst + (jj * PPW) * kB) = tot;
        } else {
          if (t.pix_ok) {
            if (dg_store)
              a.depth_grad[t.pix * D + d] = dvox;
            else if (dg_own)
              a.depth_grad[t.pix * D + d] += dvox;
            else
              atomic_add(a.depth_grad + t.pix * D + d, dvox);
          }
        }
      } else {
        dacc += dvox;
      }
    }
    if constexpr (LPP > 1) {
      wave_sync();
      if (DG && per_voxel_depth) {
        const int d = d0 + t.cl;
        if (d < d_hi && t.pix_ok) {
          const R tot = lds_at<R>(smem, q1, kDst);
          if (dg_store)
            a.depth_grad[t.pix * D + d] = tot;
          else if (dg_own)
            a.depth_grad[t.pix * D + d] += tot;
          else
            atomic_add(a.depth_grad + t.pix * D + d, tot);
        }
        wave_sync();
      }
    }
  }
  // the runs still open, then everything the windows hold
#pragma unroll
  for (int n = 0; n < NV; ++n) {
    if (__ballot(cur[n] >= 0 && cell[n].y >= 0) != 0ull) end_spread_runs(n, cur[n] >= 0);
    if (cur[n] >= 0) take_run(n);
    if (cur[n] >= 0)
      window_add<VEC, LPP, false, kForm, GAP>((unsigned)cell[n].x, cell[n].y, sg[n], ref,
                           s_data + n * WN::SLOTS * WN::STRIDE, s_tags, t.lane, t.cl);
  }
  wave_sync();
#pragma unroll
  for (int n = 0; n < NV; ++n)
    window_flush_all<VEC, LPP, kForm>(oy[n], ox[n], s_data + n * WN::SLOTS * WN::STRIDE, gview[n], srcW,
                               t.lane, tagged_slots(LPP) ? tagged_rows<VEC, LPP, kForm>(s_tags, t.lane) : wave_or(ring_rows[n]),
                               cm);
  wave_sync();  // the next view clears the window
  }  // views of the group

  // pixel-owned gradients: one store when this workgroup saw every depth, otherwise one
  // atomic add per depth segment into the zero-filled outputs
  R *rg;
  if constexpr (kWide) rg = a.ref_grad_acc;
  else rg = a.ref_grad;
  const bool single = g.nseg * g.ngroups == 1;
  if constexpr (CORR == 4) {
    // no reference image, no gradient for it
  } else if (single) {
    // (16-bit storage too: the finished sums go straight to the output, the fp32 image of
    // ref_grad is neither written nor narrowed afterwards)
    if (t.pix_ok && ch_ok) store_vec<S, VEC, false, GAP>(a.ref_grad + t.pix * C + ch0, racc);
  } else if (t.pix_ok && ch_ok) {
#pragma unroll
    for (int c = 0; c < VEC; ++c) atomic_add(rg + t.pix * C + ch0 + c / 2 * GAP + c % 2, racc[c]);
  }
  if (DG && !per_voxel_depth) {
    const R tot = group_sum<LPP>(dacc);
    if (t.cl == 0 && t.pix_ok) {
      if (single)
        a.depth_grad[t.pix] = tot;
      else
        atomic_add(a.depth_grad + t.pix, tot);
    }
  }
}

// ---- host side -------------------------------------------------------------------------------
// Depth segments: enough workgroups to fill 256 CUs several times over while every segment
// keeps at least 16 hypotheses for the register-resident taps to pay off.
inline int choose_segments(int64_t tiles, int64_t D, int lpp, int64_t target_units, bool row_sums) {
  int nseg = 1;
  // (sums in channel order: three waves per SIMD and long chunks, so the last round of workgroups is
  // the one to keep short: five views, 108 x 126 x 77, 147 -> 129 us; for the others shorter segments
  // load more taps again: f16 groups, four views, 237 x 315 x 24, 147 -> 171 us)
  const int64_t least = row_sums ? 8 : 16, min_len = lpp > least ? lpp : least;
  while (nseg < 8 && tiles * nseg < target_units && D / (nseg * 2) >= min_len) nseg *= 2;
  // a problem that does not even give every SIMD one wave: shorter segments still
  const int64_t short_len = lpp > 4 ? lpp : 4;
  while (nseg < 16 && tiles * nseg < 1024 && D / (nseg * 2) >= short_len) nseg *= 2;
  return nseg;
}

template <int LPP>
inline Geometry make_geometry(int64_t B, int64_t H, int64_t W, int64_t D, int sub, int ngroups = 1,
                              int vper = 0, bool tall = false, bool row_sums = false, bool many_taps = false,
                              bool open_lines = false) {
  constexpr int PPW = 64 / LPP;
  Geometry g;
  g.hw = (int)(H * W);
  if (PPW == 1) {
    g.tiles_x = (int)W;
    g.tiles_per_image = g.hw;
  } else {
    const int TH = tile_rows(PPW, tall), TW = PPW / TH;
    g.tiles_x = (int)((W + TW - 1) / TW);
    g.tiles_per_image = g.tiles_x * (int)((H + TH - 1) / TH);
  }
  const int64_t tiles = B * g.tiles_per_image;
  g.ngroups = ngroups;
  g.vper = vper;
  // twenty waves per SIMD over the launch: the tail of a launch with fewer is measurable
  g.nseg = choose_segments(tiles * ngroups, D, LPP, 256 * 4 * 20, row_sums);
  // A forward launch below two waves per SIMD lasts as long as its longest wave, and a segment costs
  // it nothing but the set-up: segments down to one chunk (32 channels in 8 groups, five views, 32 x 32 x 5:
  // 12.6 -> 9.9 us; samples of 8 channels, four views, 22 x 26 x 17: 10.7 -> 7.5 us; double, 8
  // channels, four views, 182 x 245 x 12: 47 -> 38 us; at four waves per SIMD a correlation of 32
  // double channels, six views, 120 x 131 x 23, is slower: 191 -> 202 us).
  // many_taps: five and six views that hold a set of taps each run two waves per SIMD at most, so a launch
  // of more than 2048 waves goes in two rounds; one that has a wave for every SIMD is left as it is (minimum
  // of CostAggregate, 8 channels, six views, 135 x 181 x 24, 782 tiles: 2 segments 37 us, 3 segments 43;
  // samples of six views, 32 channels, 44 x 62 x 107, 352 tiles: 5 segments 52 us, 7 58).
  // open_lines (see the launcher): not cut at all.
  if (vper == 0 && !open_lines && tiles * g.nseg < (many_taps ? 1024 : 2048)) {
    const int64_t chunks = (D + LPP - 1) / LPP, want = many_taps ? 2048 / tiles : (2048 + tiles - 1) / tiles;
    g.nseg = (int)(want < chunks ? want : chunks);
  }
  const int per_seg = (int)((D + g.nseg - 1) / g.nseg);
  g.seg = ((per_seg + LPP - 1) / LPP) * LPP;
  // Segments are whole chunks.  Rounded up they can be twice what was asked for (135 hypotheses of
  // 64 channels: eight segments of 17 become five of 32); a launch with fewer than two waves per
  // SIMD rounds down instead: its time is that of its longest wave (forward: best pair of 64
  // channels, six views, 16 x 21 x 135, 183 -> 99 us; group correlation bf16, 21 x 26 x 117, 25.4 ->
  // 15.5 us; gradients up to 1.6x: group correlation of 32 channels, 37 x 49 x 28, 27 -> 17 us).
  // A gradient (vper > 0) pays for every segment, so it rounds up where that costs more than the
  // longest wave: where the segments and views that add to one pixel's gradient become many (six
  // views, 105 hypotheses of 32 channels: 13 us rounded up, 18 down), and where the waves no longer
  // all run side by side -- two or three per SIMD, one where a wave has 16 pixels and more and most
  // segments would be a single chunk (one view of 16 channels, 36 x 46 x 55: 14 and 17 us).
  // Measured on 140 launches either side of these lines.
  if (g.nseg > 1 && per_seg > LPP && tiles * ngroups * ((D + g.seg - 1) / g.seg) < 2048) {
    const int down = per_seg / LPP * LPP;
    const int64_t n = (D + down - 1) / down;
    const int64_t most = LPP >= 16 ? 3072 : LPP >= 8 ? 2400 : n <= 5 ? 2048 : 1024;
    if (vper == 0 || (ngroups * n <= 35 && tiles * ngroups * n <= most)) g.seg = down;
  }
  g.nseg = (int)((D + g.seg - 1) / g.seg);
  g.total_units = tiles * g.nseg * g.ngroups;
  g.units_per_seg = (unsigned)(tiles * g.ngroups);
  // backward: runs of 32 units (the view groups of a tile are neighbours and mostly share
  // a run, hence an L2)
  // Forward: one band of tiles per XCD.  Its workgroups go to the CUs in turn, so two segments of a
  // tile that follow each other in the launch put all first segments on every other CU, all second
  // ones on the rest; where the last segment is a short one half of the chip then waits for the other
  // half (minimum of CostAggregate, 32 channels, four views, 135 x 181: 17, 20, 24 and 31 depths in
  // segments of 16 all took 59 us).  A launch whose last segment is shorter than three quarters of the
  // others goes segment by segment and ends on the short ones (17 and 20 depths 59 -> 39 us, 24 60 -> 40
  // us; group correlation, six views, 114 x 117 x 21, 38 -> 34 us).  Segments about as long as each other
  // stay beside each other: they share the lines of the output in which one ends and the next begins.
  // So do those of narrow pixels (up to eight channels) at any length: their waves write pieces of a few
  // bytes (CostAggregate of 8 channels, 326 x 430 x 82, 83 -> 140 us segment by segment), and the second
  // order costs their kernels two registers (six views of that op lost a wave per SIMD: 27 -> 42 us).
  const int64_t last = D - (int64_t)(g.nseg - 1) * g.seg;
  const bool by_segment = vper == 0 && g.nseg > 1 && LPP >= 4 && 4 * last <= 3 * (int64_t)g.seg;
  g.xcd_shift = vper > 0 ? 5 : by_segment ? kBandsBySegment : kBands;
  g.units_per_xcd = ((by_segment ? tiles : g.total_units) + 7) / 8;
  const int64_t round_to = vper > 0 ? (int64_t)8 << g.xcd_shift : 8;
  g.grid = vper > 0     ? (g.total_units + round_to - 1) / round_to * round_to
           : by_segment ? g.units_per_xcd * 8 * g.nseg
                        : g.units_per_xcd * 8;
  g.sub = sub;
  g.stream_halves = false;
  g.src_h_max = g.src_w_max = 0.f;  // set by the launcher from the source image size
  return g;
}

template <typename S>
inline bool aligned16(const S *p) {
  return (reinterpret_cast<uintptr_t>(p) & 15u) == 0;
}

}  // namespace tiled
}  // namespace chop
