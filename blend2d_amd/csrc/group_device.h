// What a tile group of a box-only band starts from.
#pragma once

#include <stdint.h>

#include "device_types.h"
#include "raster_device.h"

namespace b2amd {

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
