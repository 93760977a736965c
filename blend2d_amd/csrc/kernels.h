// Launch interface of the fill-path kernels (kernels.hip), used by the host
// frontend (context.cpp).
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include "device_types.h"
#include "lut_device.h"

namespace b2amd {

// Device views of one flush ("frame") of recorded commands.
struct FrameDev {
  const DevCanvas* canvases; uint32_t n_canvases;
  const DevCmd* cmds; uint32_t n_cmds;
  const CmdXform* xforms;
  const SrcSeg* src; uint32_t n_src;
  const double* vtx;
  const DevStyle* styles;
  const uint32_t* luts;
  uint32_t dither;         // some style samples a dithered gradient (64-bit table)
  const DevImage* images;
  uint32_t n_tiles;
  uint32_t n_groups;       // tile groups: up to 4 consecutive tiles of one band
  uint32_t n_bands;        // bands over all canvases
  uint32_t n_boxes;        // box fills among the commands
  uint64_t n_mat;          // (band, cmd) matrix entries over all canvases
  double tol_sq;           // squared flattening tolerance in 24.8 units
};

// Where a command's segments are binned: its cell in the first band, the
// distance to the next band's and the number of bands.
struct CmdBin { uint32_t row, step, bands; };
constexpr uint32_t kBoxMark = 0x80000000u;

// A line (n = 2) or a monotonic piece of a curve (n = 3, 4) that crosses the
// clip box.
struct ClipItem {
  double p[8];   // x, y
  uint32_t cmd, n;
};

// Device counters of a frame (words of FrameScratch::counters), zero at the
// start: pool flags, an error flag and the scan totals, then the cursors of
// the segment buffer's and the clip list's regions and the composited-pixel counters, each in a
// 128-byte line of its own (same-line atomics queue behind each other).
constexpr uint32_t kCounterFlags = 3, kCounterErr = 4;
constexpr uint32_t kCounterBinned = 8, kCounterList = 9;   // totals of the (band, command) cells
constexpr uint32_t kCounterTiles = 10;   // analytic tiles, then fast, solid and general box groups
constexpr uint32_t kSegRegions = 16, kCursorStep = 32, kCounterCursors = 32;
constexpr uint32_t kPixelStep = 32, kCounterPixels = kCounterCursors + 2 * kSegRegions * kCursorStep;
constexpr uint32_t kCounterWords = kCounterPixels + 64 * kPixelStep;
// What launch_report writes: the first words of the counters, the cursors and
// the pixel total.
constexpr uint32_t kReportCursors = 16, kReportClip = kReportCursors + kSegRegions,
                   kReportPixels = kReportClip + kSegRegions, kReportWords = kReportPixels + 2;

// Scratch buffers the pipeline needs; sized by the caller.
struct FrameScratch {
  uint32_t* counters;      // kCounterWords
  CmdBounds* bounds;       // n_cmds
  CmdBin* cmd_bin;         // n_cmds
  // Edge segments, in seg_regions regions of seg_stride slots: region r holds
  // min(cursor r, seg_stride) segments from slot r * seg_stride on.
  DevSeg* segs;
  uint32_t* seg_cmd;
  uint32_t* seg_rank;      // number of a segment of one band within its cell
  uint32_t* seg_cursor;    // kSegRegions cursors, then as many of the clip list, kCursorStep words apart (in counters)
  uint32_t seg_regions, seg_stride;
  // Clip list, in seg_regions regions of clip_stride slots likewise.
  ClipItem* clip;
  uint32_t clip_stride;
  uint32_t* mat_cnt;       // n_mat: segments within the cell's band
  uint32_t* mat_off;       // n_mat + 1
  uint32_t* mat_pres;      // n_mat: segments that cross bands, kBoxMark set by a box fill; later the
                           // scatter cursors of the former
  uint32_t* list_off;      // n_mat + 1
  // Per listed (band, command) cell:
  uint32_t* list_cols;     // n_list: tile-column range, first | last << 16
  uint4* list_ent;         // n_list: {command, binned offset, binned count, kMeta* bits}; boxes:
                           // {command, x0 | x1 << 16, 0, kMeta* bits}
  uint32_t* list_style;    // n_list: solid colour, or the style index of another kind of style
  DevSeg* binned;          // n_binned
  uint32_t* scan_tmp;      // scan_tmp_words()
  // Tiles of bands with analytic fills, tile groups of bands with solid box
  // fills only and tile groups of the other box-only bands, each compacted in
  // band order: exclusive scans of the per-band counts (totals at [n_bands]).
  uint32_t* band_nonsolid; // n_bands: a box fill with a non-solid style touches the band
  uint32_t* band_slow;     // n_bands: a box fill other than a solid SRC_OVER / SRC_COPY aligned box on a
                           // 32-bit canvas touches the band
  uint32_t* tile_off;      // n_bands + 1
  uint32_t* fgroup_off;    // n_bands + 1: tile groups of bands with fast box fills only
  uint32_t* sgroup_off;    // n_bands + 1
  uint32_t* ggroup_off;    // n_bands + 1
  uint4* tile_hdr;         // <= n_tiles: {canvas, band list begin, band list end, tile column | band << 16}
  uint4* group_hdr;        // <= 2 n_groups: two header words per box tile group (see group_setup),
                           // the solid bands' groups first
  // Failed fills: per command the kFailInvalidGeometry / kFailTooManySegments
  // bits of its sources (the command's segments are not binned), and one
  // word set when any command failed.
  uint32_t* cmd_err;       // n_cmds
  uint32_t* err_any;       // 1 (in counters)
  // Pool mode (sizes predicted ahead of time; null / 0 otherwise):
  uint32_t* flags;         // bit 0: segment pool overflow, bit 1: bin pool overflow (in counters)
  uint32_t binned_cap;     // capacity of `binned`
  // Work queue of the analytic tiles (k_render_queue; null otherwise):
  uint32_t* queue;         // <= n_tiles: tile slots in queue order (null: band order)
  uint32_t* queue_head;    // 1: next queue position
  uint32_t* queue_hist;    // kQueueBuckets: bucket sizes, then bucket cursors
  uint32_t* tile_key;      // <= n_tiles: bucket of each slot
  float* tile_feat;        // <= n_tiles x 16: tile cost-model features
  uint32_t* tile_cycles;   // <= n_tiles: logged wall-clock ticks per slot (null: not logged)
};

// What the compositor branches on, one word per list entry: CmdKind in bits
// 0-1, then at these bits ExecOp (3), alpha (8), even-odd (1), FetchKind (3)
// and the source format (2).
constexpr uint32_t kMetaOp = 2, kMetaAlpha = 5, kMetaEvenOdd = 13, kMetaFetch = 14, kMetaFmt = 17,
                   kMetaRow0 = 20, kMetaRow1 = 25;   // boxes: rows of the band [row 0, row 1), 5 bits each

size_t scan_tmp_words(void);

// Counters, failure bits, bounds, cell counts, box marks and band flags.
void launch_frame_init(const FrameDev& f, const FrameScratch& s, hipStream_t st);
// Writes what the host reads of the counters to pinned memory (kReportWords).
void launch_report(const FrameScratch& s, uint32_t* report, hipStream_t st);

// Stage 1: edge building, one pass over the sources into the segment buffer.
// `regions`: how many regions the buffer must be divided into.
struct EdgePlan { uint32_t batch, blocks, regions; };
EdgePlan edge_plan(uint32_t n_src);
void launch_edges(const FrameDev& f, const FrameScratch& s, hipStream_t st);
// Stage 2: binning of segments into (band, command) cells (`n_segs`: an upper
// bound of the segments) and marking of the box fills' cells; scans of the
// cells and of the bands' tile and group counts; then, once the list buffers
// are there, lists, scatter cursors and tile and group headers; and the
// scatter.
void launch_bin_count(const FrameDev& f, const FrameScratch& s, uint64_t n_segs, hipStream_t st);
void launch_scans(const FrameDev& f, const FrameScratch& s, hipStream_t st);
void launch_setup(const FrameDev& f, const FrameScratch& s, hipStream_t st);
void launch_bin_scatter(const FrameDev& f, const FrameScratch& s, uint64_t n_segs, hipStream_t st);
// Stage 3: tile rasterization + fetch + composite (n_a analytic tiles, n_f
// fast, n_s solid-box and n_g other box tile groups, or upper bounds of them).
// `strips`: workgroups per analytic tile (1, 2 or 4).
void launch_render(const FrameDev& f, const FrameScratch& s, uint32_t n_a, uint32_t strips, uint32_t n_f, uint32_t n_s, uint32_t n_g,
                   hipStream_t st);
// Work-queue form of the analytic-tile render: features of the (at most n_a)
// analytic tiles, the queue sorted by predicted cost (`pred`: the tile cost
// model's outputs, n_a x 2, or null for the segment-count heuristic), and
// the persistent render over the queue with `grid` workgroups, `wgs_per_cu`
// of them per CU (s.queue null: band order).  Box tile groups still go through launch_render.
void launch_tile_features(const FrameDev& f, const FrameScratch& s, uint32_t n_a, hipStream_t st);
void launch_tile_queue(const FrameDev& f, const FrameScratch& s, uint32_t n_a, const float* pred, hipStream_t st);
void launch_render_queue(const FrameDev& f, const FrameScratch& s, uint32_t grid, uint32_t wgs_per_cu, hipStream_t st);

void launch_fill_u32(uint32_t* p, uint32_t v, size_t n, hipStream_t st);
// Fills the gradient tables of `n_jobs` jobs (one workgroup per table).
void launch_gradient_luts(const lut::Job* jobs, const lut::Stop* stops, uint32_t n_jobs, uint32_t* luts, hipStream_t st);

// The device scratch region of bl_amd_context_replay_noalloc on device
// `dev`: its address (looked up once per device) and size in bytes.
hipError_t noalloc_scratch(int dev, void** ptr, size_t* bytes);

}  // namespace b2amd
