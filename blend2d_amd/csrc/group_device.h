// Which kernel takes a band, and what its tile groups start from.
#pragma once

#include <stdint.h>

#include "device_types.h"
#include "raster_device.h"

namespace b2amd {

// The kernels in the order of their counts: analytic fills go to the tile
// kernel, box fills to the compositor of solid SRC_OVER / SRC_COPY aligned boxes
// on 32-bit canvases, of other solid ones, or of all.
enum BandClass : uint32_t { kBandTiles = 0, kBandFast = 1, kBandSolid = 2, kBandGeneral = 3, kBandEmpty = 4 };

// `listed`: commands in the band's list.  A band without any belongs to no
// kernel: the fast compositor, which what follows would give it to, reads words,
// four times the bytes that a row of an A8 canvas has.
B2AMD_HD BandClass band_class(uint32_t listed, bool analytic, bool nonsolid, bool slow) {
  if (listed == 0u) return kBandEmpty;
  if (analytic) return kBandTiles;
  return nonsolid ? kBandGeneral : slow ? kBandSolid : kBandFast;
}

// Whether the canvas's first command copies an opaque colour over all of the
// canvas's pixels [x0, x1) x [y0, y1), so that what they held doesn't matter.
// A canvas without commands has no first one: `cmd_base` is then the next
// canvas's, or one past the last command of the frame.
B2AMD_HD bool starts_opaque(const DevCanvas& cv, const DevCmd* cmds, const DevStyle* styles, uint32_t x0, uint32_t y0,
                            uint32_t x1, uint32_t y1) {
  if (cv.n_cmds == 0u) return false;
  const DevCmd& c = cmds[cv.cmd_base];
  if (c.kind != kCmdBoxA || c.alpha != 255u || (c.op != kOpSrcCopy && c.op != kOpSrcOver)) return false;
  if (c.box[0] > (int32_t)x0 || c.box[1] > (int32_t)y0 || c.box[2] < (int32_t)x1 || c.box[3] < (int32_t)y1) return false;
  const DevStyle& s = styles[c.style];
  return s.kind == kFetchSolid && (c.op == kOpSrcCopy || (s.solid >> 24) == 255u);
}

}  // namespace b2amd
