// Which calls that the tile-shaped kernels could serve keep a lane per channel because it is the faster
// one (the strip kernels; CostVolumeV3 with more than 16 groups: a thread per voxel).  Only double has
// such calls: its tiles need twice the registers and run two waves per SIMD, and its lane-per-channel
// kernels are held to four.  Times in microseconds, lane per channel against tiles, as "12 : 15".
#pragma once

#include "internal.h"

namespace chop {

template <typename S>
bool lanes_are_faster(const Args<S> &a, bool backward) {
  if (sizeof(S) != 8) return false;
  const int64_t lpp = a.C > 16 && a.C < 32 ? 8 : a.C / 4;  // lanes of a pixel
  const bool few_tiles = a.pixels() * lpp / 64 < 2048;
  if (backward) {
    // Gradients of group correlation over a few depths: clearing and writing back a workgroup's window
    // costs the same for two depths as for a whole chunk, and wide pixels share it between few pixels.
    // The line: 3/4 depth per lane of a pixel.  64 channels, two views, 200 x 260: 4 depths 246 : 436, 8
    // depths 415 : 595; three views, 90 x 100: 4 depths 100 : 146, 12 depths 166 : 161.  32 channels,
    // three views, 138 x 151: 2 depths 140 : 175, 4 depths 190 : 200, 6 depths 227 : 219.  16 channels: 2
    // depths 77 : 83, 4 depths 108 : 93.  Where the tiles do not fill the chip the launch is bound by
    // latency and the tiles' shorter chains win up to 32 channels (five views, 60 x 80, 600 tiles: 32
    // channels, 2 depths 45 : 38), but not at 64 (70 : 89).
    // The minimum at 64 channels at any depth: each view's workgroups pass over the other views' voxels
    // with four pixels to a wave.  200 x 260, four views: 12 depths 1001 : 1455, 32 depths 1833 : 2454,
    // one hypothesis field 1421 : 1622; two views, 32 depths 1109 : 1224, one hypothesis field 886 : 842.
    if (a.corr == GROUP_CORRELATION &&
        ((4 * a.D < 3 * lpp && (lpp == 16 || !few_tiles)) || (lpp == 16 && a.reduce != 0)))
      return true;
    // One view over a few depths, few tiles: narrow pixels have only the clearing and writing back to do
    // (38 x 40 x 6, 8 channels: group correlation 10.6 : 13.6, squared differences 8.5 : 11.9; 16 channels
    // 16.6 : 16.3).
    return a.N == 1 && lpp <= 2 && a.D < 12 && few_tiles &&
           (a.corr == GROUP_CORRELATION || a.corr == SQUARED_DIFFERENCE);
  }
  // Squared differences of many views, or of 64 channels and three views in launches of few tiles.
  return a.corr == SQUARED_DIFFERENCE && ((lpp >= 8 && a.N >= 5) || (lpp == 16 && a.N >= 3 && few_tiles));
}

}  // namespace chop
