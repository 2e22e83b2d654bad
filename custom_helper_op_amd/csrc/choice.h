// Which calls that the tile-shaped kernels could serve keep a lane per channel because it is the faster
// one (the strip kernels; CostVolumeV3 with more than 16 groups: a thread per voxel).  A lane per channel
// spreads a depth over more lanes and needs fewer registers, so it wins where a launch is bound by the chain
// of steps in one wave and not by work.  Times in microseconds, lane per channel against tiles, as
// "12 : 15"; float64 where nothing else is said.
#pragma once

#include "internal.h"

namespace chop {

template <typename S>
int64_t lanes_of_a_pixel(const Args<S> &a) {
  return a.C > 16 && a.C < 32 ? 8 : a.C / 4;
}

// Values, in double or with idle lanes (20, 24 and 28 channels in any type).  A tile's wave takes a chunk of
// as many depths as a pixel has lanes through every view, one view's taps after the other's: until every
// SIMD has a wave of its own, a launch takes as long as one wave, and the chain grows with the views.
//   waves  32 channels, squared differences:  three views, 190 (38 x 40 x 6) 7.8 : 11.1, 570 10.5 : 14.8,
//          950 14.8 : 14.9, 1050 (50 x 56 x 24) 18.4 : 17.6, 1800 23.7 : 17.5; two views, 190 6.5 : 7.5,
//          380 7.7 : 8.9, 570 10.2 : 9.8; one view, 120 5.5 : 6.1, 190 5.6 : 5.3, 570 7.7 : 6.8.  24 channels
//          in float32, three views: 570 9.9 : 12.1, 1200 15.2 : 13.3.
//   16 channels leave each lane half as many chains: squared differences, three views, 364 8.4 : 9.3, 600
//   10.3 : 9.8; group correlation 200 8.5 : 9.8, 546 11.5 : 10.5.  8 channels: tiles at any size.
//   CostAggregate and FeatureAggregate hold less per view (four views, 32 channels: with differences 180
//   12.5 : 13.2, 380 14.7 : 16.0, 700 16.7 : 16.5; samples alone 380 12.2 : 16.4, 570 18.2 : 17.9).
// Few depths shorten the tiles' chain, not the lanes' (one view, 38 x 40: 3 depths 5.4 : 4.5; CostAggregate,
// four views, 64 channels, 20 x 24: 3 depths 13.4 : 9.7; samples of 16 channels, six views, 19 x 20: one depth
// 10.3 : 7.3; group correlation of 32 channels, six views, 58 x 61: 4 depths 19.3 : 15.2).  Not with the
// squared differences of five and six views (64 channels, 19 x 21, one depth 6.2 : 9.1).
template <typename S>
bool lanes_are_faster_forward(const Args<S> &a) {
  const bool idle_lanes = a.C > 16 && a.C < 32;
  if ((sizeof(S) != 8 && !idle_lanes) || a.corr == BEST_GROUP_PAIR) return false;
  const int64_t lpp = lanes_of_a_pixel(a), tiles = a.pixels() * lpp / 64;
  const int64_t waves = tiles * ((a.D + lpp - 1) / lpp);
  if (lpp <= 2) {
    // One view's minimum at 8 channels writes and does next to nothing else.  Where the volume is far beyond
    // the caches the strips' rows go out faster: group correlation, 200 x 260, 48 depths 65.7 : 76.1, 333 x
    // 390, 24 depths 79.1 : 104 (200 x 260, 24 depths 42.1 : 36.4); squared differences, 200 x 260, 86 depths
    // 149 : 182 (100 x 130, 86 depths 58.8 : 57.8).
    return lpp == 2 && a.N == 1 && a.reduce != 0 &&
           ((a.corr == GROUP_CORRELATION && waves >= 32768) ||
            (a.corr == SQUARED_DIFFERENCE && waves >= 65536));
  }
  // (one view's minimum of 28 channels likewise, 160 x 200: 96 depths 0.83 of the tiles' time, 32 depths 1.06)
  if (sizeof(S) == 8 && idle_lanes && a.corr == SQUARED_DIFFERENCE && a.reduce != 0 && a.N == 1 && waves >= 40960)
    return true;
  // Two waves of the squared differences' minimum of many views fit a SIMD: a little over 2048 tiles leave a
  // second round nearly empty, until the depths can be cut to fill it (five views, 32 channels, 2400 tiles:
  // 12 depths 64.5 : 72.4, 24 depths 101 : 115, 48 depths 189 : 172; 3250 tiles, 12 depths 83.4 : 73.8).
  if (a.corr == SQUARED_DIFFERENCE && a.reduce != 0 && a.N >= 5 && lpp >= 8 && tiles > 2048 &&
      tiles <= 2560 && a.D <= 24)
    return true;
  const bool one_value = a.corr == SUM_SQUARED_DIFFERENCE, samples = a.corr == WARP_ONLY;
  int64_t line;
  if (lpp == 4)
    line = one_value || a.N == 1 ? 0 : (a.corr == SQUARED_DIFFERENCE ? 512 : 256) / (a.N == 2 ? 2 : 1);
  else if (one_value)
    line = a.N == 1 ? 0 : a.N == 2 ? 192 : 384;
  else
    line = a.N == 1 ? 192 : a.N == 2 || samples || (a.corr == GROUP_CORRELATION && a.D < 5) ? 384 : 768;
  if (waves >= line) return false;
  if (one_value) return 2 * a.D >= lpp;
  return a.D >= 4 || (a.D == 3 && a.N >= 3 && !samples) ||
         (a.corr == SQUARED_DIFFERENCE && a.N >= 5 && lpp >= 8);
}

// Gradients in double of one view, or of two, in launches that leave most of the chip idle.  With so few
// depths to a tile there is little to share in its window, and clearing it, collecting in it and writing it
// back is a longer chain than the strips' atomic additions.  The line is a number of tiles times depths; it
// lies higher for the gradients with one value per voxel (their strips read less) and for wide pixels (whose
// tiles are small).  One view, 38 x 40 x 6, squared differences: 4 channels 9.7 : 14.4, 8 channels 10.1 :
// 13.4, 32 channels 13.5 : 15.3, 64 channels 15.7 : 21.4; beyond the line 60 x 80 x 24, 8 channels 17.6 :
// 17.6, 60 x 80 x 6, 32 channels 21.2 : 18.0, 60 x 80 x 12, 64 channels (1200 tiles) 45.6 : 34.9; with one
// value per voxel 90 x 110 x 6, 8 channels 14.2 : 19.0, x 12 23.4 : 19.4.  Not group correlation of 32
// channels (38 x 40 x 6 17.5 : 16.4) or its minimum of 64.  16 channels: tiles (38 x 40 x 12 15.0 : 11.4).
// Two views, squared differences: 4 channels, 38 x 40 x 6 12.8 : 15.6, 60 x 80 x 12 22.1 : 17.6; 64 channels,
// 20 x 24 x 12 17.6 : 22.3, 38 x 40 x 12 29.2 : 27.2.
template <typename S>
bool lanes_are_faster_few_tiles(const Args<S> &a) {
  const int64_t lpp = lanes_of_a_pixel(a), tiles = a.pixels() * lpp / 64, steps = tiles * a.D;
  if (a.corr == BEST_GROUP_PAIR || a.N > 2 || tiles >= 512) return false;
  if (a.D < 3) return a.corr == SUM_SQUARED_DIFFERENCE && a.N == 1 && lpp == 2;
  const bool correlation = a.corr == GROUP_CORRELATION;
  if (a.N == 2)
    return lpp == 1    ? steps < (correlation && a.reduce == 0 ? 256 : 1024) && a.D < 16 && (a.D > 3 || tiles >= 128)
           : lpp == 16 ? steps < 3072
                       : false;
  return lpp <= 2    ? steps < (a.corr == SUM_SQUARED_DIFFERENCE ? 2048 : correlation && a.reduce != 0 ? 2560 : 1024)
         : lpp == 8  ? steps < 2560 && !correlation
         : lpp == 16 ? steps < 8192 && !(correlation && a.reduce != 0)
                     : false;
}

// Gradients of group correlation in double.  Over a few depths: a workgroup clears its window and writes it
// back once for two depths as for a whole chunk, and the minimum passes over every view's voxels to find its
// own, of which wider groups have fewer.  Groups of four channels, 200 x 260 and planes
// from depth 2 on unless something else is given; the strips' time goes up with the depths and the number of groups, the tiles' hardly.
//   Mean   64 channels, two views: 2 depths 261 : 343, 3 depths 370 : 423, 4 depths 487 : 461; four views:
//          3 depths 736 : 853, 4 depths 955 : 910, 38 x 45 x 1 23 : 30.  32 channels, four views: 2 depths 281 :
//          319, 3 depths 401 : 371.  16 channels, four views: 3 depths 157 : 182, 4 depths 189 : 193, and with
//          1200 tiles (120 x 160) 71 : 65.
//          4 channels, whose window is one texel column to a lane: long sweeps, from 0.7 of the tiles' time
//          (planes from depth 5 on, 96 depths, four views) to 0.9 (planes from 0.7); 32 depths 0.85 and 1.56.
//   Minimum at 64 channels, two views and more: at any depth, as a wave holds four pixels.  Two views: 4
//          depths 248 : 437, 12 depths 585 : 718; four views, 12 depths 1003 : 1464, 32 depths 1833 : 2454.
//          One view has nothing to pass over: 4 depths 223 : 187.
//   Minimum at 32 channels, four views: groups of one and two, 2 depths 0.81 and 0.74 of the tiles' time, 4
//          depths 1.21 and 1.02; of four, 4 depths 246 : 346, 8 depths 415 : 432; of eight, 6 depths 0.80, 8 depths
//          0.92.  Six views: 2 depths 0.78, 60 x 80 x 4 1.06; groups of eight, 200 x 260 x 6 0.96.  Three views:
//          4 depths 253 : 274, 6 depths 312 : 318, 60 x 80 x 4 41 : 37.
//   Minimum at 16 channels: two views 3 depths 96 : 104, 4 depths 112 : 110; four views 153 : 186, 179 : 192.
//   Minimum at 8 channels: groups of one and two, four views, 8 depths 1.2 and 1.0 of the tiles' time, planes
//          from 5 on and 330 x 400 1.56 and 1.25; of four 132 : 139, 12 depths 191 : 177; 120 x 160 x 8 57 :
//          65; 60 x 80 x 4 26 : 22; of eight, 8 depths 0.61 to 0.85, 16 depths 0.77 to 0.97.  Six views, groups
//          of four: 188 : 199, but 120 x 160 x 8 88 : 77.  Two views, any groups: 60 x 80 x 12 20.6 : 22.9, x 16
//          0.9, 120 x 160 x 8 0.9.  One view: 120 x 160 x 8 21.4 : 24.8, x 16 0.9, 200 x 260 x 8 44.8 : 40.2.
//   Minimum at 4 channels: three views, 8 depths 76 : 121, 12 depths 113 : 148; 32 depths, two views, groups of
//          one 0.75 to 1.15, of two 0.72 to 1.06, of four 0.70 to 0.91 of the tiles' time; 96 depths 0.6 to 0.75
//          with any; 16 depths, groups of four, two views and more 0.76 to 0.99.  One view, 8 depths, 120 x
//          160 0.76 and 0.94, 330 x 400 0.91 and 1.68.  Four views, 60 x 80 x 8 25.5 : 22.9, 120 x 160 x 8 44 : 51.
template <typename S>
bool lanes_are_faster_correlation(const Args<S> &a) {
  const int64_t lpp = lanes_of_a_pixel(a), tiles = a.pixels() * lpp / 64, sub = a.C / a.groups;
  if (a.reduce == 0) {
    if (lpp == 1) return a.D >= 64 && tiles >= 256;
    if (lpp == 16 && a.N > 1 && a.D <= 2) return tiles >= 256;
    return a.N > 1 && lpp >= 4 && a.D < (lpp == 8 ? 3 : 4) && tiles >= (lpp == 16 ? 1024 : 2048);
  }
  switch (lpp) {
    case 16: return a.N > 1;
    case 8:
      if (a.N >= 4 && a.D <= 2) return tiles >= 256;
      if (a.N == 4) return a.D <= (sub == 1 ? 2 : sub == 2 ? 4 : 8) && tiles >= 256;
      if (a.N > 4) return sub > 1 && a.D <= 2 + (sub < 8 ? sub : 6) && tiles >= 2048;
      return a.N > 1 && a.D <= 4 && tiles >= 2048;
    case 4: return a.N > 1 && a.D <= 3 && tiles >= 2048;
    case 2:
      if (a.N <= 2 && tiles < 1024) return a.D <= (tiles < 256 ? 16 : 8) && a.D > (a.N == 1 || tiles >= 256 ? 1 : 3);
      if (a.N == 1 || sub < 4) return false;
      return a.D <= (sub == 8 && a.N <= 4 && tiles >= 1024 ? 16 : 8) && tiles >= 256 * (a.N - 2);
    default:
      if (a.D >= 64) return tiles >= 256;
      if (a.D > 12) return tiles >= 256 && (a.D >= 24 ? sub > 1 || a.N == 1 : a.N > 1 && (sub == 4 || (sub == 2 && a.N >= 4)));
      if (a.D <= 1 || tiles < 64 * (a.N - 2)) return false;
      return a.N == 1 ? tiles < 512 : a.D > 2 && (sub == 4 || (sub == 2 && a.D <= 8));
  }
}

// Gradients in double over one to eight depths of the ops without groups, and of CostVolumeV3 (see above: the
// window's cost is that of a chunk).  At 64 channels a workgroup has four pixels to share its window, with
// idle lanes eight of fewer channels.  As a part of the tiles' time, 200 x 260 unless another size is given:
//   Squared differences, 64 channels, two and four views: one depth 0.79 and 0.77, two depths 1.01 and 0.99;
//   minimum 0.70 and 0.63, two depths 0.84 and 0.75, three 1.03.  24 channels, two views: 0.75, two depths
//   0.84, three 0.99, but 60 x 80 x 2 1.09.  32 channels and fewer: even at one depth.
//   CostAggregate's mean: the same.  Its minimum passes over every view's voxels: 64 channels, two views, two
//   depths 0.79, four 1.00; three views, four 0.88, eight 1.15; four views, eight 0.91, 60 x 80 x 8 0.93,
//   twelve 1.02; 24 channels, four views, four 0.77, eight 0.94; three views four 0.94 (120 x 160 1.05); 32
//   channels, four views only, four 0.89; 8 channels, two to four views, two depths 0.79 to 0.87.
//   CostVolumeV3's mean, up to 16 groups: 64 channels, groups of eight, two views, eight depths 0.79, three
//   views 0.92, four views, four depths 0.93; of four, two views, four depths 0.82, three views 0.92, four
//   views, two depths 0.92; 32 channels, two and four views, one depth 0.80 and 0.74, two 0.92 and 0.98; 16
//   channels, one depth 0.82 and 0.71, two 0.98 and 0.93.
template <typename S>
bool lanes_are_faster_few_depths(const Args<S> &a) {
  const int64_t lpp = lanes_of_a_pixel(a), tiles = a.pixels() * lpp / 64;
  const bool idle_lanes = a.C > 16 && a.C < 32, low = a.reduce != 0, one_value = a.corr == SUM_SQUARED_DIFFERENCE;
  if (a.N < 2 || a.D > 8 || tiles < 512) return false;
  if (a.corr == BEST_GROUP_PAIR) {
    if (a.groups > 16 || a.N > 4 || low) return false;
    if (lpp == 16) return tiles >= 4096 && a.D * a.N <= (a.C == 8 * a.groups ? 16 : 8);
    return (lpp == 8 && a.D <= 2 && tiles >= 4096) || (lpp == 4 && a.D == 1 && tiles >= 2048);
  }
  if (a.corr != SQUARED_DIFFERENCE && !one_value) return false;
  if (one_value && low) {
    if (lpp == 16) return a.D <= (a.N == 2 ? 2 : a.N == 3 ? 5 : 8);
    if (idle_lanes) return a.D <= (a.N <= 3 ? 3 : 5) && tiles >= 2048;
    return a.N <= 4 && ((lpp == 8 && a.N == 4 && a.D <= 4 && tiles >= 2048) || (lpp == 2 && a.D <= 2 && tiles >= 1024));
  }
  return lpp == 16 ? a.D <= (low ? 2 : 1) : idle_lanes && a.D <= 2 && tiles >= 2048;
}

// Gradients of CostVolumeV3's minimum.  One source group and one reference group of one view receive the
// voxel's gradient, and the mask names them: nothing is searched for, and next to nothing is added up.  The
// tiles' workgroup of each view still walks every voxel with all of a pixel's lanes and clears and writes
// back its window; their work grows with the views times the channels, that of the others hardly.  Groups of
// four and eight channels in float run the tiles at any size.
//   More than 16 groups: a thread per voxel.  Its time is that of a few additions to memory, so the line is a
//   number of depths per view.  Float, 200 x 260 unless another size is given: 32 channels in groups of one,
//   two views, 8 depths 113 : 138, 12 depths 147 : 158, 32 depths 350 : 265; four views, 12 depths 144 : 215;
//   one view 4 depths 46 : 48, 12 depths 116 : 79; 383 x 534 x 27, two views, planes from depth 0.7, 2 and 5 on
//   1123 : 1492, 1138 : 1107 and 1126 : 851, and 300 x 400 x 27, four views, 683 : 1117, 693 : 921, 696 : 764.  64 channels in groups of one, two views, 8 depths 119 :
//   223, 32 depths 375 : 455; one view, 32 depths 316 : 287.  64 channels in groups of two, four views, 8
//   depths 210 : 340; two views 211 : 224, one view, 4 depths 91 : 81.  Few tiles, 20 x 24: 32 channels, two
//   views, 12 depths 8 : 18, 32 depths 13 : 18.  Double: the tiles take twice the time and more.  64
//   channels in groups of one, four views, 8 depths 124 : 638; in groups of two 217 : 644; 32 channels, two
//   views, 8 depths 103 : 208, 32 depths 330 : 484, 120 x 160 x 96 353 : 375.
//   Up to 16 groups: a lane per channel.  It has no window to clear.  One view of 8 channels, 60 x 80 x 12 13 :
//   15, x 32 24 : 16.  32 channels in groups of two, float: four views, 4 depths 70 : 95, 12 depths even; two
//   views, 383 x 534 x 4 0.87 of the tiles' time; 20 x 24 x 12 10 : 14.  Double: four views, 8 depths 266 :
//   326, two views, 8 depths 239 : 208 (four views' texel cache is the largest that the strips hold).  64
//   channels in groups of four and eight, double: four views, 60 x 80 x 12 56 : 72, 200 x 260 x 4 296 : 515,
//   60 x 80 x 96 293 : 239; six views, 4 depths 504 : 612, 120 x 160 x 12 353 : 319; one view 4 depths 1.26 of
//   the tiles' time.  16 channels, float, four views, 383 x 534: 4 depths 0.76 of the tiles' time, 12 depths
//   1.09; double: tiles.
template <typename S>
bool lanes_are_faster_best_pair(const Args<S> &a) {
  const bool wide = sizeof(S) == 8;
  const int64_t lpp = lanes_of_a_pixel(a), tiles = a.pixels() * lpp / 64, sub = a.C / a.groups;
  if (a.reduce == 0 || (!wide && sub >= 4)) return false;
  if (a.groups > 16) {
    if ((tiles < 1024 && a.D <= 12) || (tiles < 256 && a.D <= (wide ? 160 : sub == 1 ? 64 : 32))) return true;
    if (wide) return a.groups == 64 || a.D < (sub == 1 ? 64 * a.N - 32 : 32 * a.N - 12);
    return sub == 1 ? a.D <= (lpp == 16 ? 16 : a.N == 1 ? 6 : 9) * a.N : a.N > 1 && a.D <= 5 * a.N;
  }
  switch (lpp) {
    case 2:
      return (a.N == 1 && tiles < 256 && a.D <= 16) ||
             (wide && a.N > 1 && a.N <= 4 && a.D <= (tiles >= 4096 ? 7 : 3) && tiles >= 1024);
    case 4:
      if (wide) return a.N > 1 && a.D == 1 && tiles >= 2048;
      return (a.N == 1 && tiles < 64 && a.D <= 16) || (a.N > 1 && tiles >= 8192 && a.D <= 6);
    case 8:
      if (tiles < 128) return a.D >= 8 && a.D <= 16 && a.N <= 4;
      if (!wide) return a.N > 1 && a.D <= 6 && tiles >= (a.N >= 4 ? 768 : 2048);
      if (a.N == 2 || a.N == 3) return a.D <= 2 && tiles >= 4096;
      return a.N >= 4 && ((a.D <= 4 && tiles >= 512) || (a.N == 4 && a.D <= 12 && tiles >= 1024));
    default: return a.N > 4 ? a.D <= 6 && tiles >= 1024 : a.N > 2 ? a.D <= 32 : a.N > 1 && a.D <= 24;
  }
}

template <typename S>
bool lanes_are_faster(const Args<S> &a, bool backward) {
  if (!backward) return lanes_are_faster_forward(a);
  if (a.corr == BEST_GROUP_PAIR && lanes_are_faster_best_pair(a)) return true;
  if (sizeof(S) != 8) return false;
  return lanes_are_faster_few_tiles(a) || lanes_are_faster_few_depths(a) ||
         (a.corr == GROUP_CORRELATION && lanes_are_faster_correlation(a));
}

}  // namespace chop
