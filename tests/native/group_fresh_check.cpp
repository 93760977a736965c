// Checks which kernel takes a band and which tile groups start from an opaque
// colour (blend2d_amd/csrc/group_device.h, compiled here for the host).  The command
// and style tables end where a page without access begins, and the command
// behind the last one, where there is room for one, is a stale one whose style
// lies far outside its table: a canvas that recorded nothing must not lead to
// either.
//
//   group_fresh_check      exit status 0 when all agree, "mismatches N"
#include <stdint.h>
#include <stdio.h>
#include <string.h>
#include <sys/mman.h>
#include <unistd.h>

#include "../../blend2d_amd/csrc/group_device.h"

using namespace b2amd;

namespace {

// `n` objects ending at a page without access.
template<typename T>
T* guarded(size_t n) {
  const size_t page = (size_t)sysconf(_SC_PAGESIZE), bytes = (n * sizeof(T) + page - 1) / page * page;
  uint8_t* p = (uint8_t*)mmap(nullptr, bytes + page, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS, -1, 0);
  if (p == MAP_FAILED || mprotect(p + bytes, page, PROT_NONE)) _exit(3);
  return (T*)(p + bytes - n * sizeof(T));
}

DevCmd box(uint32_t op, uint32_t alpha, uint32_t style, int x0, int y0, int x1, int y1) {
  DevCmd c;
  memset(&c, 0, sizeof(c));
  c.kind = kCmdBoxA;
  c.op = op;
  c.alpha = alpha;
  c.style = style;
  c.box[0] = x0; c.box[1] = y0; c.box[2] = x1; c.box[3] = y1;
  return c;
}

int bad = 0;
void expect(const char* what, bool got, bool want) {
  if (got == want) return;
  fprintf(stderr, "%s: got %d, want %d\n", what, got, want);
  bad++;
}

}  // namespace

int main() {
  DevStyle* styles = guarded<DevStyle>(3);
  memset(styles, 0, 3 * sizeof(DevStyle));
  styles[0].kind = kFetchSolid; styles[0].solid = 0xFF102030u;
  styles[1].kind = kFetchSolid; styles[1].solid = 0x80102030u;
  styles[2].kind = kFetchLinear;

  DevCanvas cv;
  memset(&cv, 0, sizeof(cv));
  cv.w = 300; cv.h = 40; cv.n_cmds = 1;
  const struct { const char* what; DevCmd cmd; bool want; } cases[] = {
    {"opaque over", box(kOpSrcOver, 255, 0, 0, 0, 300, 40), true},
    {"translucent over", box(kOpSrcOver, 255, 1, 0, 0, 300, 40), false},
    {"translucent copy", box(kOpSrcCopy, 255, 1, 0, 0, 300, 40), true},
    {"copy at half alpha", box(kOpSrcCopy, 128, 0, 0, 0, 300, 40), false},
    {"plus", box(kOpPlus, 255, 0, 0, 0, 300, 40), false},
    {"gradient", box(kOpSrcCopy, 255, 2, 0, 0, 300, 40), false},
    {"a column short on the right", box(kOpSrcOver, 255, 0, 0, 0, 299, 40), false},
    {"a column short on the left", box(kOpSrcOver, 255, 0, 257, 0, 300, 40), false},
    {"the group's columns only", box(kOpSrcOver, 255, 0, 256, 0, 300, 40), true},
    {"a row short", box(kOpSrcOver, 255, 0, 0, 0, 300, 39), false},
    {"from the group's first row", box(kOpSrcOver, 255, 0, 0, 32, 300, 40), true},
    {"from a row below it", box(kOpSrcOver, 255, 0, 0, 33, 300, 40), false},
  };
  DevCmd* cmds = guarded<DevCmd>(2);
  for (const auto& k : cases) {
    cmds[0] = k.cmd;
    // the last group of the last band: columns 256 .. 299, rows 32 .. 39
    expect(k.what, starts_opaque(cv, cmds, styles, 256, 32, 300, 40), k.want);
  }

  // canvases without commands: between two others, and last
  DevCanvas none = cv;
  none.n_cmds = 0;
  cmds[0] = box(kOpSrcCopy, 255, 0, 0, 0, 300, 40);
  cmds[1] = box(kOpSrcCopy, 255, 0x40000000u, 0, 0, 300, 40);   // stale
  none.cmd_base = 0;
  expect("empty canvas before another", starts_opaque(none, cmds, styles, 0, 0, 256, 16), false);
  none.cmd_base = 1;
  expect("empty canvas before stale memory", starts_opaque(none, cmds, styles, 0, 0, 256, 16), false);
  none.cmd_base = 2;
  expect("empty canvas at the end of the table", starts_opaque(none, cmds, styles, 0, 0, 256, 16), false);

  // bands: every class, and none without a command
  expect("paths", band_class(3, true, false, false) == kBandTiles, true);
  expect("paths over a gradient", band_class(3, true, true, true) == kBandTiles, true);
  expect("solid boxes", band_class(1, false, false, false) == kBandFast, true);
  expect("solid boxes on A8", band_class(1, false, false, true) == kBandSolid, true);
  expect("gradient boxes", band_class(1, false, true, true) == kBandGeneral, true);
  expect("no commands", band_class(0, false, false, false) == kBandEmpty, true);

  printf("mismatches %d\n", bad);
  return bad ? 1 : 0;
}
