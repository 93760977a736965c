// Fill-path kernels for gfx950.
//
//   edges    source segments (line / quad / cubic) taken by lanes as they get
//            free: transform, clip, split, flatten -> 24.8 edge segments, in
//            one pass.
//   bin      per segment: number within its (band, command) cell, scatter;
//            per band a compacted, submission-ordered list of the commands
//            touching it.
//   render   one 256-thread workgroup per 64x16 tile (or strip of it): the
//            destination is loaded once into registers, every command of
//            the band is rasterized into LDS cells with LDS atomics, turned
//            into coverage by a per-scanline DPP scan, fetched, composited
//            in submission order, and the tile is stored once.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "device_types.h"
#include "edge_device.h"
#include "group_device.h"
#include "kernels.h"
#include "pipe_device.h"
#include "raster_device.h"

#include <mutex>

namespace b2amd {

// ---------------------------------------------------------------------------
// Utilities
// ---------------------------------------------------------------------------

// Scratch of the execution that allocates nothing
// (bl_amd_context_replay_noalloc): every intermediate buffer of a frame is a
// slice of this region.  Each device holds its own copy for the life of the
// process; every call on a device shares it, so calls that overlap on one
// device race (the library's flushes and replays are serialized by its
// device queue).
//
// Its size: a segment takes 24 bytes with the number it is binned by, a piece of
// a curve 72, against 20 and 88 when segments were counted in a pass of their
// own.  A frame takes at most 1.2 times what it took then, so all that fitted
// 64 MiB fits here.
constexpr size_t kNoAllocScratchBytes = (size_t)80 << 20;
static __device__ __align__(256) uint8_t scratch[kNoAllocScratchBytes];

hipError_t noalloc_scratch(int dev, void** ptr, size_t* bytes) {
  constexpr int kMaxDevices = 64;
  static std::mutex mu;
  static void* addr[kMaxDevices] = {};
  if (dev < 0 || dev >= kMaxDevices) return hipErrorInvalidDevice;
  std::lock_guard<std::mutex> lock(mu);
  if (!addr[dev]) {
    // the array's host-side name is not a device address: look the address
    // up on this device (current) and use only that
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return e;
    addr[dev] = p;
  }
  *ptr = addr[dev];
  *bytes = kNoAllocScratchBytes;
  return hipSuccess;
}

__global__ void k_fill_u32(uint32_t* p, uint32_t v, size_t n) {
  size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

void launch_fill_u32(uint32_t* p, uint32_t v, size_t n, hipStream_t st) {
  if (!n) return;
  hipLaunchKernelGGL(k_fill_u32, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, p, v, n);
}

// Everything a frame starts from, in one launch: counters and cursors, command
// failure bits and bounds, the (band, command) counts, presence flags and band
// flags.
__global__ void k_frame_init(FrameDev f, FrameScratch s) {
  const size_t i0 = (size_t)blockIdx.x * blockDim.x + threadIdx.x, step = (size_t)gridDim.x * blockDim.x;
  for (size_t i = i0; i < kCounterWords; i += step) s.counters[i] = 0u;
  for (size_t i = i0; i < f.n_cmds; i += step) {
    s.cmd_err[i] = 0u;
    s.bounds[i] = CmdBounds{INT32_MAX, INT32_MIN, INT32_MAX, INT32_MIN};
    const DevCanvas& cv = f.canvases[f.cmds[i].canvas];
    s.cmd_bin[i] = CmdBin{(uint32_t)cv.mat_base + (uint32_t)i - cv.cmd_base, cv.n_cmds, cv.bands};
  }
  for (size_t i = i0; i < f.n_mat; i += step) {
    s.mat_cnt[i] = 0u;
    s.mat_pres[i] = 0u;
  }
  for (size_t i = i0; i < f.n_bands; i += step) {
    s.band_nonsolid[i] = 0u;
    s.band_slow[i] = 0u;
  }
}

void launch_frame_init(const FrameDev& f, const FrameScratch& s, hipStream_t st) {
  const uint64_t n = std::max<uint64_t>({kCounterWords, f.n_cmds, f.n_mat, f.n_bands});
  hipLaunchKernelGGL(k_frame_init, dim3((unsigned)std::min<uint64_t>((n + 255) / 256, 4096)), dim3(256), 0, st, f, s);
}

// The counters the host reads, into pinned memory: one small launch instead of
// a copy per value.  `report` layout: kReport* words.
__global__ __launch_bounds__(64) void k_report(FrameScratch s, uint32_t* report) {
  const uint32_t lane = threadIdx.x;
  const unsigned long long* px = (const unsigned long long*)(s.counters + kCounterPixels);
  unsigned long long sum = px[lane * (kPixelStep / 2)];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o, 64);
  if (lane < kReportCursors) report[lane] = s.counters[lane];
  if (lane < 2 * kSegRegions) report[kReportCursors + lane] = s.counters[kCounterCursors + lane * kCursorStep];
  if (lane == 0) {
    report[kReportPixels] = (uint32_t)sum;
    report[kReportPixels + 1] = (uint32_t)(sum >> 32);
  }
}

void launch_report(const FrameScratch& s, uint32_t* report, hipStream_t st) {
  hipLaunchKernelGGL(k_report, dim3(1), dim3(64), 0, st, s, report);
}

// One gradient table per workgroup, every entry computed on its own
// (lut_device.h).  The stops of a job were validated and sorted on the
// host (offsets in [0, 1], n >= 1), so every position lies in [0, size).
__global__ void __launch_bounds__(256) k_gradient_luts(const lut::Job* __restrict__ jobs,
                                                       const lut::Stop* __restrict__ stops,
                                                       uint32_t* __restrict__ luts) {
  const lut::Job j = jobs[blockIdx.x];
  const lut::Stop* st = stops + j.stop0;
  if (j.wide) {
    for (uint32_t e = threadIdx.x; e < j.size; e += 256u) {
      const uint64_t v = lut::entry64(st, j.n_stops, j.size, e);
      luts[(size_t)j.lut + 2u * e] = (uint32_t)v;
      luts[(size_t)j.lut + 2u * e + 1u] = (uint32_t)(v >> 32);
    }
    return;
  }
  for (uint32_t e = threadIdx.x; e < j.size; e += 256u) luts[(size_t)j.lut + e] = lut::entry(st, j.n_stops, j.size, e);
}

void launch_gradient_luts(const lut::Job* jobs, const lut::Stop* stops, uint32_t n_jobs, uint32_t* luts, hipStream_t st) {
  if (!n_jobs) return;
  hipLaunchKernelGGL(k_gradient_luts, dim3(n_jobs), dim3(256), 0, st, jobs, stops, luts);
}

// ---------------------------------------------------------------------------
// Wave helpers
// ---------------------------------------------------------------------------

// Cross-lane moves on the VALU (DPP): lanes without a source keep `old`.
template<int kCtrl, int kRowMask>
__device__ __forceinline__ uint32_t dpp(uint32_t old, uint32_t v) {
  return (uint32_t)__builtin_amdgcn_update_dpp((int)old, (int)v, kCtrl, kRowMask, 0xF, false);
}

// Inclusive prefix sum (maximum) within groups of W = 16, 32 or 64 lanes, all
// lanes active: row shifts by 1, 2, 4 and 8, then the last lane of a row (of
// 16) added to the next row, of the lower half to the upper.
template<int W>
__device__ __forceinline__ uint32_t lane_scan_add(uint32_t v) {
  v += dpp<0x111, 0xF>(0u, v);
  v += dpp<0x112, 0xF>(0u, v);
  v += dpp<0x114, 0xF>(0u, v);
  v += dpp<0x118, 0xF>(0u, v);
  if (W >= 32) v += dpp<0x142, 0xA>(0u, v);
  if (W >= 64) v += dpp<0x143, 0xC>(0u, v);
  return v;
}
__device__ __forceinline__ uint32_t wave_scan_max(uint32_t v) {
  v = max(v, dpp<0x111, 0xF>(0u, v));
  v = max(v, dpp<0x112, 0xF>(0u, v));
  v = max(v, dpp<0x114, 0xF>(0u, v));
  v = max(v, dpp<0x118, 0xF>(0u, v));
  v = max(v, dpp<0x142, 0xA>(0u, v));
  v = max(v, dpp<0x143, 0xC>(0u, v));
  return v;
}
// LDS written by lanes of this wave is visible to its other lanes after this
// (a wave's LDS operations execute in order; the fence holds the compiler).
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
}
__device__ __forceinline__ uint32_t lane_value(uint32_t v, uint32_t lane) {
  return (uint32_t)__builtin_amdgcn_readlane((int)v, (int)lane);
}

// ---------------------------------------------------------------------------
// Stage 1: edges
// ---------------------------------------------------------------------------

__device__ __forceinline__ edge::P xform_pt(const CmdXform& m, const double* vtx, uint32_t i) {
  double x = vtx[2 * (size_t)i], y = vtx[2 * (size_t)i + 1];
  if (m.scale_only) return edge::P{x * m.m00 + m.m20, y * m.m11 + m.m21};
  return edge::P{x * m.m00 + y * m.m10 + m.m20, x * m.m01 + y * m.m11 + m.m21};
}

__device__ __forceinline__ edge::Clip canvas_clip(uint32_t size) {
  edge::Clip clip;
  clip.x0 = 0.0; clip.y0 = 0.0;
  clip.x1 = (double)(size & 0xFFFFu) * 256.0;
  clip.y1 = (double)(size >> 16) * 256.0;
  clip.ix0 = (int32_t)clip.x0;
  clip.ix1 = (int32_t)clip.x1;
  return clip;
}

// A failed source fails its whole command (rare; the plain stores race
// benignly, every writer sets the same bits).
__device__ __forceinline__ void fail_cmd(const FrameScratch& s, uint32_t cmd, uint32_t bits) {
  atomicOr(&s.cmd_err[cmd], bits);
  *s.err_any = 1u;
}

// What a lane keeps of the command whose sources it is working on.
struct LaneBounds {
  uint32_t cmd;
  int32_t min_x, max_x, min_y, max_y;
  __device__ __forceinline__ void reset(uint32_t c) { cmd = c; min_x = min_y = INT32_MAX; max_x = max_y = INT32_MIN; }
  __device__ __forceinline__ void add(int32_t x0, int32_t y0, int32_t x1, int32_t y1) {
    const int32_t lo = min(x0, x1) >> 8, hi = max(x0, x1) >> 8;
    min_x = min(min_x, lo);
    max_x = max(max_x, hi);
    min_y = min(min_y, y0);
    max_y = max(max_y, y1);
  }
};

// Segments of one wave of k_edges_clip on their way out: staged in LDS and
// written to the wave's region of the segment buffer with coalesced stores,
// one atomic on the region's cursor per flush.
constexpr uint32_t kEdgeStage = 512;
// Parts of curves that lie inside the clip box, found by lanes in their walk
// across it: the whole wave flattens them afterwards.
constexpr uint32_t kInnerList = 64;
struct EdgeStage {
  DevSeg seg[kEdgeStage];
  uint32_t cmd[kEdgeStage];
  double inner[8][kInnerList];         // the four points (x, y)
  uint32_t inner_cmd[kInnerList];
  uint32_t inner_how[kInnerList];      // sign | points << 1
};
struct EdgeOut {
  EdgeStage& stage;
  const FrameScratch& s;
  uint32_t* cursor;
  size_t region;
  uint32_t staged;   // uniform
  __device__ __forceinline__ EdgeOut(EdgeStage& st, const FrameScratch& scratch, uint32_t wid)
      : stage(st), s(scratch), cursor(scratch.seg_cursor + wid % scratch.seg_regions * kCursorStep),
        region((size_t)(wid % scratch.seg_regions) * scratch.seg_stride), staged(0) {}
  // All lanes call it.
  __device__ __forceinline__ void flush() {
    if (!staged) return;
    const uint32_t lane = threadIdx.x & 63u;
    wave_sync();
    uint32_t base = 0;
    if (lane == 0) base = atomicAdd(cursor, staged);
    base = (uint32_t)__builtin_amdgcn_readfirstlane((int)base);
    for (uint32_t i = lane; i < staged; i += 64u) {
      const uint32_t pos = base + i;
      if (pos < s.seg_stride) {
        s.segs[region + pos] = stage.seg[i];
        s.seg_cmd[region + pos] = stage.cmd[i];
      }
    }
    if (s.flags && lane == 0 && base + staged > s.seg_stride) atomicOr(s.flags, 1u);
    staged = 0;
    wave_sync();
  }
};

// Emitter of what a lane runs to completion on its own (sources that cross
// the clip box): a staging slot per segment, or a slot of the region itself
// once the stage is full.
struct ClipEmit {
  EdgeOut& out;
  uint32_t* count;   // of staged segments, then of inner parts
  LaneBounds& bd;
  __device__ __forceinline__ bool give(const edge::P* p, int n, uint32_t sign) {
    const uint32_t at = atomicAdd(count + 1, 1u);
    if (at >= kInnerList) return false;
    EdgeStage& st = out.stage;
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const edge::P q = p[i == 3 ? n - 1 : i];
      st.inner[2 * i][at] = q.x;
      st.inner[2 * i + 1][at] = q.y;
    }
    st.inner_cmd[at] = bd.cmd;
    st.inner_how[at] = sign | (uint32_t)n << 1;
    return true;
  }
  __device__ __forceinline__ void push(int32_t x0, int32_t y0, int32_t x1, int32_t y1, uint32_t sign) {
    const DevSeg g{x0, y0, (int32_t)((uint32_t)x1 | (sign << 31)), y1};
    bd.add(x0, y0, x1, y1);
    const uint32_t at = atomicAdd(count, 1u);
    if (at < kEdgeStage) {
      out.stage.seg[at] = g;
      out.stage.cmd[at] = bd.cmd;
      return;
    }
    const uint32_t pos = atomicAdd(out.cursor, 1u);
    if (pos < out.s.seg_stride) {
      out.s.segs[out.region + pos] = g;
      out.s.seg_cmd[out.region + pos] = bd.cmd;
    }
    else if (out.s.flags) atomicOr(out.s.flags, 1u);
  }
};

// Wave-wide minimum of a signed value (the identity INT32_MAX where a lane has
// nothing to say), all lanes active; the maximum is ~min(~v).
__device__ __forceinline__ int32_t wave_min(int32_t v) {
  const int id = INT32_MAX;
  v = min(v, (int32_t)dpp<0x111, 0xF>((uint32_t)id, (uint32_t)v));
  v = min(v, (int32_t)dpp<0x112, 0xF>((uint32_t)id, (uint32_t)v));
  v = min(v, (int32_t)dpp<0x114, 0xF>((uint32_t)id, (uint32_t)v));
  v = min(v, (int32_t)dpp<0x118, 0xF>((uint32_t)id, (uint32_t)v));
  v = min(v, (int32_t)dpp<0x142, 0xA>((uint32_t)id, (uint32_t)v));
  v = min(v, (int32_t)dpp<0x143, 0xC>((uint32_t)id, (uint32_t)v));
  return (int32_t)lane_value((uint32_t)v, 63u);
}

// Folds the bounds of the lanes in `who` into their commands, one set of
// atomics per distinct command of the wave (all lanes call it).
__device__ __forceinline__ void fold_bounds(CmdBounds* __restrict__ bounds, uint64_t who, const LaneBounds& b) {
  const uint32_t lane = threadIdx.x & 63u;
  while (who) {
    const uint32_t cmd = lane_value(b.cmd, (uint32_t)__builtin_ctzll(who));
    const bool in = ((who >> lane) & 1ull) && b.cmd == cmd;
    const int32_t mnx = wave_min(in ? b.min_x : INT32_MAX), mny = wave_min(in ? b.min_y : INT32_MAX);
    const int32_t mxx = ~wave_min(in ? ~b.max_x : INT32_MAX), mxy = ~wave_min(in ? ~b.max_y : INT32_MAX);
    if (lane == 0 && mnx <= mxx) {
      CmdBounds* bd = &bounds[cmd];
      atomicMin(&bd->min_x, mnx);
      atomicMax(&bd->max_x, mxx);
      atomicMin(&bd->min_y, mny);
      atomicMax(&bd->max_y, mxy);
    }
    who &= ~__ballot(in);
  }
}

// Lanes that have just halved their root keep the first half as theirs and
// hand the other to lanes that wait (all lanes call it).  True for a lane that
// got one, its bounds being those of the curve's command then; before(other)
// is called by all lanes, `other` where a lane changes its command.
template<typename B, typename Before>
__device__ __forceinline__ bool share_halves(edge::CurveWalk<B>& w, uint32_t* giver, bool halved, bool waits, LaneBounds& bd,
                                             CmdBounds* bounds, Before&& before) {
  const uint32_t lane = threadIdx.x & 63u;
  const uint64_t below = (1ull << lane) - 1ull;
  const uint64_t give = __ballot(halved), idle = __ballot(waits);
  if (!give || !idle) return false;
  const uint32_t n = min((uint32_t)__popcll(give), (uint32_t)__popcll(idle));
  const bool gives = halved && (uint32_t)__popcll(give & below) < n;
  const uint32_t rank = (uint32_t)__popcll(idle & below);
  const bool takes = waits && rank < n;
  if (gives) giver[__popcll(give & below)] = lane;
  wave_sync();
  const int from = takes ? (int)giver[rank] : (int)lane;
  wave_sync();
  const uint32_t cmd = (uint32_t)__shfl((int)bd.cmd, from, 64);
  const uint32_t how = (uint32_t)__shfl((int)(w.sign | (uint32_t)w.root.n << 1), from, 64);
  const bool other = takes && cmd != bd.cmd;
  before(other);
  const uint64_t fold = __ballot(other && bd.cmd != 0xFFFFFFFFu);
  if (fold) fold_bounds(bounds, fold, bd);
  if (other) bd.reset(cmd);
  edge::P half[4];
#pragma unroll
  for (int i = 0; i < 4; i++) half[i] = edge::P{__shfl(w.top[i].x, from, 64), __shfl(w.top[i].y, from, 64)};
  if (takes) w.start(half, (int)(how >> 1), how & 1u);
  if (gives) {
#pragma unroll
    for (int i = 0; i < 4; i++) w.root.p[i] = w.m.p[i];
    w.level = w.path = 0;
  }
  return takes;
}

// Source segments -> 24.8 edge segments, in one pass.
//
// A curve of ten segments next to one of a single segment leaves most lanes
// waiting when every lane flattens its own, and the pieces, counts and
// segments of separate passes cross HBM several times.  Here a wave walks
// `batch` consecutive sources: a lane that is done takes the next one, splits
// it into monotonic pieces as it gets to them and flattens a step per turn of
// the wave's loop (test, then split or emit), so lanes stay busy whatever
// their curves need; only segments go to memory.  Taking sources and pieces is
// done for many waiting lanes at once.
//
// The subdivision has no stack: a per-lane stack lives in scratch memory, far
// more than the caches hold, and its traffic was what bounded the kernel (2.9
// ms on the glyph frame below).  The right half of the
// last split is kept in registers; any other node is split again from the
// piece along its path, which repeats the same arithmetic and so gives the
// same points.
//
// A source that crosses the clip box goes to the clip list, whole lines or the
// monotonic pieces of a curve: its walk is long and branchy, and k_edges_clip
// gives every piece a lane.  A piece inside the box is finite and at most 65535
// pixels across, and each split cuts its distance from its chord to a quarter,
// so it is flat after about ten: the limits of the general builder cannot be
// reached here.
//
// Each lane stages up to four segments in LDS; a flush writes them lane by
// lane, so the segments of a contour stay together (binning gathers equal
// cells among neighbours), at the cursor of the wave's region (s.seg_regions
// of s.seg_stride slots each): one counter takes 11.4 ns per atomic on this
// chip, sixteen take 1.2 together.  Slots past the stride are counted but not
// written: the caller reads the cursors and grows the buffer, or (pool mode)
// the overflow flag is raised.
//
// Measured against splitting, counting and writing in passes of their own
// (clip list included): 1024 glyph canvases, 5.1 million quads into 18.3
// million segments, 3.12 -> 1.18 ms; 10 000 cubic paths, 2.8 million segments,
// 0.82 -> 0.58.
//
// Few long curves would leave most of a wave's lanes without work and be one
// serial chain each.  Once a wave has no sources left, a lane that halves its
// root (the piece, or what is left of it when nothing waits above the node in
// hand) keeps the first half and hands the other to a waiting lane: the nodes
// and their points are the same whichever lane gets to them, and the order of
// segments doesn't matter.  With it, clip list not included: 32 uneven canvases
// 380 -> 100 us, 10 000 cubic paths 418 -> 213, 2000 pattern shapes 65 -> 29,
// a frame of panels 64 -> 27.
constexpr uint32_t kLaneStage = 4;
struct EdgeWave {
  DevSeg seg[kLaneStage][64];
  double cv[8][64];    // each lane's source curve, transformed (x, y)
  double cut[8][64];   // parameters it is cut at, then 1
  uint32_t giver[64];  // lanes that hand half of their node over
};

__global__ __launch_bounds__(256) void k_edges(FrameDev f, FrameScratch s, uint32_t batch) {
  __shared__ EdgeWave waves[4];
  using B = edge::Builder<ClipEmit>;
  const uint32_t lane = threadIdx.x & 63u;
  const uint64_t below = (1ull << lane) - 1ull;
  const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const uint32_t wid = blockIdx.x * 4u + wave, n_waves = gridDim.x * 4u;
  EdgeWave& ws = waves[wave];
  const uint32_t region_i = wid % s.seg_regions;
  const size_t region = (size_t)region_i * s.seg_stride;
  uint32_t* const cursor = s.seg_cursor + region_i * kCursorStep;

  // lane state
  enum : uint32_t { kIdle, kPiece, kFlat };
  uint32_t mode = kIdle;
  uint32_t staged = 0;
  LaneBounds bd;
  bd.reset(0xFFFFFFFFu);
  edge::P at{0.0, 0.0};          // end point of the last piece
  double t_cut = 0.0;
  int n_cuts = 0, cut_i = 0;
  int points = 3;
  edge::CurveWalk<B> walk;
  walk.root.n = walk.m.n = 3;
  walk.sign = 0;
  bool crossing = false;         // the curve leaves the clip box of `size`
  uint32_t size = 0;

  auto flush = [&]() {
    const uint32_t incl = lane_scan_add<64>(staged);
    const uint32_t total = lane_value(incl, 63u);
    if (!total) return;
    uint32_t base = 0;
    if (lane == 0) base = atomicAdd(cursor, total);
    base = (uint32_t)__builtin_amdgcn_readfirstlane((int)base);
    const uint32_t pos = base + incl - staged;
#pragma unroll
    for (uint32_t k = 0; k < kLaneStage; k++) {
      if (k < staged && pos + k < s.seg_stride) {
        s.segs[region + pos + k] = ws.seg[k][lane];
        s.seg_cmd[region + pos + k] = bd.cmd;
      }
    }
    if (s.flags && lane == 0 && base + total > s.seg_stride) atomicOr(s.flags, 1u);
    staged = 0;
  };
  auto put = [&](int32_t x0, int32_t y0, int32_t x1, int32_t y1, uint32_t sg) {
    ws.seg[staged++][lane] = DevSeg{x0, y0, (int32_t)((uint32_t)x1 | (sg << 31)), y1};
    bd.add(x0, y0, x1, y1);
  };

  // All lanes call it: one item of each lane that has one to the clip list.
  auto clip_put = [&](bool on, const edge::P p[4], uint32_t n) {
    const uint64_t who = __ballot(on);
    uint32_t base = 0;
    if (lane == 0) base = atomicAdd(cursor + kSegRegions * kCursorStep, (uint32_t)__popcll(who));
    base = (uint32_t)__builtin_amdgcn_readfirstlane((int)base) + (uint32_t)__popcll(who & below);
    if (!on) return;
    if (base < s.clip_stride) {
      ClipItem* const it = s.clip + (size_t)region_i * s.clip_stride + base;
#pragma unroll
      for (int i = 0; i < 4; i++) { it->p[2 * i] = p[i].x; it->p[2 * i + 1] = p[i].y; }
      it->cmd = bd.cmd;
      it->n = n;
    }
    else if (s.flags) atomicOr(s.flags, 1u);
  };

  for (uint32_t b0 = wid * batch; b0 < f.n_src; b0 += n_waves * batch) {
    uint32_t next = b0;
    const uint32_t end = f.n_src - b0 < batch ? f.n_src : b0 + batch;
    for (;;) {
      // waiting lanes take the next sources
      const uint64_t idle = __ballot(mode == kIdle);
      if (idle && next < end) {
        const uint32_t rank = (uint32_t)__popcll(idle & below);
        const bool take = mode == kIdle && next + rank < end;
        SrcSeg sg{0xFFFFFFFFu, 0, 0, 0};
        if (take) sg = f.src[next + rank];
        next += min((uint32_t)__popcll(idle), end - next);
        // a lane's staged segments and bounds belong to one command
        const bool other = take && sg.cmd != bd.cmd;
        if (__ballot((other && staged) || staged == kLaneStage)) flush();
        const uint64_t fold = __ballot(other && bd.cmd != 0xFFFFFFFFu);
        if (fold) fold_bounds(s.bounds, fold, bd);
        if (other) bd.reset(sg.cmd);
        bool to_clip = false;
        edge::P cv[4];
        if (take) {
          const CmdXform& xf = f.xforms[sg.cmd];
          const edge::Clip clip = canvas_clip(xf.canvas_size);
          const int npts = sg.kind == kSrcLine ? 2 : sg.kind == kSrcQuad ? 3 : 4;
          cv[0] = xform_pt(xf, f.vtx, sg.i0);
          cv[1] = xform_pt(xf, f.vtx, sg.i1);
          cv[2] = npts > 2 ? xform_pt(xf, f.vtx, sg.i1 + 1) : cv[1];
          cv[3] = npts > 3 ? xform_pt(xf, f.vtx, sg.i1 + 2) : cv[2];
          // A curve with a NaN or infinite control point has no defined
          // flattening (the reference subdivides it to its recursion limit
          // or trips its own assertions): the fill fails with
          // BL_ERROR_INVALID_GEOMETRY.
          bool finite = true;
          uint32_t common = 0xFu, any = 0u;
#pragma unroll
          for (int i = 0; i < 4; i++) {   // (the last point may count more than once)
            finite = finite && isfinite(cv[i].x) && isfinite(cv[i].y);
            const uint32_t fl = edge::fxy(clip, cv[i]);
            common &= fl;
            any |= fl;
          }
          int32_t lx0 = 0, ly0 = 0, lx1 = 0, ly1 = 0;   // a line's or border line's segment
          points = npts;
          if (npts == 2) {
            if (any) to_clip = true;
            else {
              lx0 = edge::trunc_i(cv[0].x); ly0 = edge::trunc_i(cv[0].y);
              lx1 = edge::trunc_i(cv[1].x); ly1 = edge::trunc_i(cv[1].y);
            }
          }
          else if (!finite) fail_cmd(s, sg.cmd, kFailInvalidGeometry);
          else if (common) {
            // above or below the canvas: nothing; left or right of it: the
            // border line over its y range (edgebuilder_p.h:1618-1890)
            if (!(common & (edge::CY0 | edge::CY1))) {
              lx0 = lx1 = common & edge::CX0 ? clip.ix0 : clip.ix1;
              ly0 = edge::trunc_i(edge::dclamp(cv[0].y, clip.y0, clip.y1));
              ly1 = edge::trunc_i(edge::dclamp(cv[3].y, clip.y0, clip.y1));
            }
          }
          else {
            if (npts == 3) {
              double c[3];
              n_cuts = B::cuts_quad(cv, c);
              if (n_cuts > 1) ws.cut[0][lane] = c[0];
              if (n_cuts > 2) ws.cut[1][lane] = c[1];
              if (n_cuts) ws.cut[n_cuts - 1][lane] = 1.0;
            }
            else {
              double c[8];
              n_cuts = B::cuts_cubic(cv, c);
              for (int i = 0; i < n_cuts; i++) ws.cut[i][lane] = c[i];
            }
#pragma unroll
            for (int i = 0; i < 4; i++) { ws.cv[2 * i][lane] = cv[i].x; ws.cv[2 * i + 1][lane] = cv[i].y; }
            cut_i = 0;
            t_cut = 0.0;
            at = cv[0];
            crossing = any != 0u;
            size = xf.canvas_size;
            mode = kPiece;
          }
          if (ly0 < ly1) put(lx0, ly0, lx1, ly1, 0u);
          else if (ly0 > ly1) put(lx1, ly1, lx0, ly0, 1u);
        }
        if (__ballot(to_clip)) clip_put(to_clip, cv, 2u);
      }

      // lanes between pieces start their next one
      if (__ballot(mode == kPiece)) {
        if (__ballot(staged == kLaneStage)) flush();
        bool to_clip = false;
        edge::P p[4];
        if (mode == kPiece) {
          const bool quad = points == 3;
          edge::P cv[4];
#pragma unroll
          for (int i = 0; i < 4; i++) cv[i] = edge::P{ws.cv[2 * i][lane], ws.cv[2 * i + 1][lane]};
          p[3] = cv[3];
          if (n_cuts == 0) {
            p[0] = cv[0]; p[1] = cv[1]; p[2] = cv[2];
          }
          else {
            double t = ws.cut[cut_i++][lane];
            if (quad) {
              B::piece_quad(cv, t_cut, t, cut_i == n_cuts, at, p);
              p[3] = p[2];
            }
            else {
              while (t == t_cut && cut_i < n_cuts) t = ws.cut[cut_i++][lane];
              B::piece_cubic(cv, t_cut, t, cut_i == n_cuts, at, p);
            }
            t_cut = t;
          }
          at = p[3];
          const uint32_t sign = p[0].y > at.y ? 1u : 0u;
          // from the top down: first and last point, and the control points
          // kept between them
          const edge::P a = sign ? p[3] : p[0], z = sign ? p[0] : p[3];
          edge::P c1 = quad ? p[1] : sign ? p[2] : p[1], c2 = quad ? z : sign ? p[1] : p[2];
          mode = kFlat;
          if (crossing) {
            DevSeg line;
            const edge::PieceWay way = edge::place_piece(canvas_clip(size), p, a, z, line);
            if (way == edge::kPieceLine) put(line.x0, line.y0, line.x1, line.y1, sign);
            to_clip = way == edge::kPieceClip;
            if (way != edge::kPieceInside) mode = cut_i == n_cuts ? kIdle : kPiece;
          }
          if (mode == kFlat) {
            const double xl = edge::dmin(a.x, z.x), xr = edge::dmax(a.x, z.x);
            const edge::P from_top[4] = {
              a, edge::P{edge::dclamp(c1.x, xl, xr), edge::dclamp(c1.y, a.y, z.y)},
              quad ? z : edge::P{edge::dclamp(c2.x, xl, xr), edge::dclamp(c2.y, a.y, z.y)}, z};
            walk.start(from_top, points, sign);
          }
        }
        if (__ballot(to_clip)) clip_put(to_clip, p, (uint32_t)points);
      }

      // flatten, a step for every lane at a time, until enough lanes wait
      for (;;) {
        const uint64_t busy = __ballot(mode == kFlat);
        if (!busy) break;
        if (__popcll(busy) < 40 && (next < end || __ballot(mode == kPiece) != 0ull)) break;
        if (__ballot(staged == kLaneStage)) flush();
        bool halved = false;
        if (mode == kFlat && !walk.step(f.tol_sq, halved, put)) mode = cut_i == n_cuts ? kIdle : kPiece;
        if (next >= end) {
          if (share_halves(walk, ws.giver, halved, mode == kIdle, bd, s.bounds, [&](bool other) {
                if (__ballot(other && staged)) flush();
              })) {
            cut_i = n_cuts = 0;
            mode = kFlat;
          }
        }
      }
      if (next >= end && __ballot(mode != kIdle) == 0ull) break;
    }
  }
  flush();
  const uint64_t have = __ballot(bd.cmd != 0xFFFFFFFFu);
  if (have) fold_bounds(s.bounds, have, bd);
}

// The clip list: lines and monotonic pieces that leave the canvas, one a lane,
// through the general builder.  What bounds it is the serial chain of the
// longest curve, so the builder only follows a curve to where it crosses the
// clip box: parts inside it are left to the wave, whose lanes share them as
// k_edges does.  Few items go one to a wave (at least 1 / 4 / 16 a wave: uneven
// canvases 64 / 75 / 129 us, 2000 pattern shapes 31 / 43 / 63, panels 26 / 30 /
// 40).  Before, a lane walked its whole curve: uneven canvases 275 -> 64 us,
// 10 000 cubic paths 163 -> 83, pattern shapes 67 -> 31, panels 38 -> 26, 1024
// glyph canvases (short curves) 311 -> 289.
__global__ __launch_bounds__(64) void k_edges_clip(FrameDev f, FrameScratch s) {
  __shared__ EdgeStage stage;
  __shared__ uint32_t count[2];
  __shared__ uint32_t giver[64];
  const uint32_t lane = threadIdx.x;
  const uint32_t r = blockIdx.x % s.seg_regions;
  const uint32_t n = min(s.seg_cursor[(kSegRegions + r) * kCursorStep], s.clip_stride);
  const ClipItem* const items = s.clip + (size_t)r * s.clip_stride;
  EdgeOut out(stage, s, r);
  LaneBounds bd;
  bd.reset(0xFFFFFFFFu);
  // few items are spread over many waves: each is a serial chain
  const uint32_t blocks = gridDim.x / s.seg_regions;
  const uint32_t per = min(64u, max(1u, (n + blocks - 1u) / blocks));
  for (uint32_t i0 = blockIdx.x / s.seg_regions * per; i0 < n; i0 += blocks * per) {
    const uint32_t i = i0 + lane;
    const bool on = lane < per && i < n;
    const uint32_t cmd = on ? items[i].cmd : 0u;
    const bool other = on && cmd != bd.cmd;
    const uint64_t fold = __ballot(other && bd.cmd != 0xFFFFFFFFu);
    if (fold) fold_bounds(s.bounds, fold, bd);
    if (other) bd.reset(cmd);
    out.flush();
    if (lane < 2u) count[lane] = 0u;
    wave_sync();
    if (on) {
      const ClipItem it = items[i];
      const edge::Clip clip = canvas_clip(f.xforms[cmd].canvas_size);
      ClipEmit emit{out, count, bd};
      edge::Builder<ClipEmit> b(emit, clip, f.tol_sq);
      const edge::P* ip = (const edge::P*)it.p;
      if (it.n == 2) b.line(ip[0], ip[1]);
      else {
        edge::P stack[edge::Builder<ClipEmit>::kLimit * 4];
        b.curve_piece(ip, (int)it.n, stack);
      }
      if (b.invalid) fail_cmd(s, cmd, b.invalid);
    }
    wave_sync();
    const uint32_t n_inner = min((uint32_t)__builtin_amdgcn_readfirstlane((int)count[1]), kInnerList);
    if (n_inner) {
      edge::CurveWalk<edge::Builder<ClipEmit>> walk;
      walk.root.n = walk.m.n = 3;
      walk.sign = 0;
      bool busy = false;
      uint32_t next = 0;
      for (;;) {
        const uint64_t idle = __ballot(!busy);
        if (idle && next < n_inner) {
          const uint32_t at = next + (uint32_t)__popcll(idle & ((1ull << lane) - 1ull));
          const bool takes = !busy && at < n_inner;
          next += min((uint32_t)__popcll(idle), n_inner - next);
          const uint32_t c = takes ? stage.inner_cmd[at] : 0u;
          const bool changes = takes && c != bd.cmd;
          const uint64_t old = __ballot(changes && bd.cmd != 0xFFFFFFFFu);
          if (old) fold_bounds(s.bounds, old, bd);
          if (changes) bd.reset(c);
          if (takes) {
            edge::P p[4];
#pragma unroll
            for (int i = 0; i < 4; i++) p[i] = edge::P{stage.inner[2 * i][at], stage.inner[2 * i + 1][at]};
            const uint32_t how = stage.inner_how[at];
            walk.start(p, (int)(how >> 1), how & 1u);
            busy = true;
          }
        }
        if (!__ballot(busy)) break;
        bool halved = false;
        if (busy)
          busy = walk.step(f.tol_sq, halved, [&](int32_t ax, int32_t ay, int32_t bx, int32_t by, uint32_t sg) {
            ClipEmit{out, count, bd}.push(ax, ay, bx, by, sg);
          });
        if (next >= n_inner && share_halves(walk, giver, halved, !busy, bd, s.bounds, [](bool) {})) busy = true;
      }
      wave_sync();
    }
    out.staged = min((uint32_t)__builtin_amdgcn_readfirstlane((int)count[0]), kEdgeStage);
  }
  out.flush();
  const uint64_t have = __ballot(bd.cmd != 0xFFFFFFFFu);
  if (have) fold_bounds(s.bounds, have, bd);
}

// Sources per wave, regions and workgroups for `n_src` sources.  A wave's
// curves are serial chains, so a small frame spreads them thin (8 a wave fill
// the chip from 32 thousand sources on); a large one gives each lane several,
// so that it has a next one to take.
EdgePlan edge_plan(uint32_t n_src) {
  EdgePlan p;
  p.batch = std::min(256u, std::max(8u, n_src / 4096u));
  const uint32_t batches = (n_src + p.batch - 1) / p.batch;
  p.blocks = std::max(1u, std::min((batches + 3) / 4, 4096u));
  p.regions = n_src >= 8192 ? kSegRegions : 1u;
  return p;
}

void launch_edges(const FrameDev& f, const FrameScratch& s, hipStream_t st) {
  if (!f.n_src) return;
  const EdgePlan p = edge_plan(f.n_src);
  hipLaunchKernelGGL(k_edges, dim3(p.blocks), dim3(256), 0, st, f, s, p.batch);
  const uint64_t most = (uint64_t)s.clip_stride * s.seg_regions;
  const uint32_t waves = (uint32_t)std::min<uint64_t>((most + 63) / 64, 8192);
  if (waves) hipLaunchKernelGGL(k_edges_clip, dim3((waves + s.seg_regions - 1) / s.seg_regions * s.seg_regions), dim3(64), 0, st, f, s);
}

// ---------------------------------------------------------------------------
// Stage 2: binning
// ---------------------------------------------------------------------------

__device__ __forceinline__ void seg_bands(const DevSeg& g, int bands, int& b0, int& b1) {
  if (g.y1 <= g.y0) { b0 = 1; b1 = 0; return; }
  int ey0 = g.y0 >> 8;
  int ey1 = (g.y1 - 1) >> 8;
  b0 = ey0 / kTileH;
  b1 = ey1 / kTileH;
  b0 = b0 < 0 ? 0 : b0;
  b1 = b1 > bands - 1 ? bands - 1 : b1;
}

// Pool mode: a segment-pool overflow (flag bit 0) leaves the frame to be
// redone with exact counting, so binning is skipped.
__device__ __forceinline__ bool pool_overflowed(const FrameScratch& s) { return s.flags && (*s.flags & 1u); }

// The binning kernels take 256 x P consecutive segments of a region at a
// time, P a thread; workgroups are dealt to the regions in turn and stride over
// a region's slots.  P is 8 (one global atomic per cell and 2048 segments)
// unless that leaves CUs idle, 1 then.  Grid over at most `n` segment slots.
constexpr uint32_t kBinPer = 8, kBinBlocks = 4096;
inline uint32_t bin_per(uint64_t n) { return n >= (uint64_t)256 * kBinPer * 256 ? kBinPer : 1u; }
inline uint32_t bin_blocks(const FrameScratch& s, uint64_t n) {
  const uint64_t tile = 256ull * bin_per(n);
  const uint32_t b = (uint32_t)std::min<uint64_t>((n + tile - 1) / tile, kBinBlocks);
  return (b + s.seg_regions - 1) / s.seg_regions * s.seg_regions;
}
struct RegionWalk {
  size_t base;               // first slot of the region
  uint32_t first, step, n;   // this workgroup's first slot, its stride, the slots used
};
__device__ __forceinline__ RegionWalk region_walk(const FrameScratch& s, uint32_t block, uint32_t blocks, uint32_t per) {
  const uint32_t r = block % s.seg_regions;
  RegionWalk w;
  w.base = (size_t)r * s.seg_stride;
  w.n = min(s.seg_cursor[r * kCursorStep], s.seg_stride);
  w.first = block / s.seg_regions * 256u * per;
  w.step = blocks / s.seg_regions * 256u * per;
  return w;
}

// Cells of one segment: the first one's index (0xFFFFFFFF: none, or its
// command failed), the distance between bands and the number of bands.
struct SegCells { uint32_t cell, step, n; };
__device__ __forceinline__ SegCells seg_cells(const FrameScratch& s, const DevSeg& g, uint32_t cmd) {
  const CmdBin cb = s.cmd_bin[cmd];
  SegCells c{0xFFFFFFFFu, cb.step, 0u};
  int b0, b1;
  seg_bands(g, (int)cb.bands, b0, b1);
  if (b1 < b0 || s.cmd_err[cmd]) return c;
  c.cell = cb.row + (uint32_t)b0 * cb.step;
  c.n = (uint32_t)(b1 - b0) + 1u;
  return c;
}

// Box fills are present in every band their box touches; a box fill with a
// non-solid style also marks its bands (they take the general compositor), one
// that k_render_box_fast does not handle (it takes aligned boxes of a solid
// colour, SRC_OVER or SRC_COPY, on 32-bit canvases) marks them slow.
// 16 threads per command, each taking every 16th band of the box.
__device__ __forceinline__ void box_presence(const FrameDev& f, const FrameScratch& s, uint32_t i) {
  const uint32_t c = i >> 4;
  if (c >= f.n_cmds) return;
  const DevCmd& cmd = f.cmds[c];
  if (cmd.kind == kCmdAnalytic) return;
  const DevCanvas& cv = f.canvases[cmd.canvas];
  const int b0 = cmd.box[1] / kTileH, b1 = (cmd.box[3] - 1) / kTileH;
  const uint64_t row = cv.mat_base + (uint64_t)(c - cv.cmd_base);
  const bool nonsolid = f.styles[cmd.style].kind != kFetchSolid;
  const bool slow = nonsolid || cmd.kind != kCmdBoxA || (cmd.op != kOpSrcOver && cmd.op != kOpSrcCopy) ||
                    cv.format == kFmtA8;
  for (int b = b0 + (int)(i & 15u); b <= b1; b += 16) {
    s.mat_pres[row + (uint64_t)b * cv.n_cmds] = kBoxMark;
    if (nonsolid) s.band_nonsolid[cv.band_base + b] = 1u;
    if (slow) s.band_slow[cv.band_base + b] = 1u;
  }
}

// Counts the segments of every cell and numbers those that stay within one
// band (the common case) in theirs.  The segments of one workgroup fall into a
// few cells, contours being contiguous, so they are counted in an LDS hash
// table first and every cell takes its range with one global atomic.  Segments
// that cross bands are counted apart (low bits of mat_pres) and take their
// places when they are scattered.  The workgroups past the first `blocks` mark
// the box fills.
template<uint32_t kPer>
__global__ __launch_bounds__(256) void k_bin_count(FrameDev f, FrameScratch s, uint32_t blocks) {
  constexpr uint32_t kSlots = 512, kNone = 0xFFFFFFFFu;
  __shared__ uint32_t key[kSlots], cnt[kSlots], at[kSlots];
  if (blockIdx.x >= blocks) {
    box_presence(f, s, (blockIdx.x - blocks) * 256u + threadIdx.x);
    return;
  }
  if (pool_overflowed(s)) return;
  const RegionWalk w = region_walk(s, blockIdx.x, blocks, kPer);
  for (uint32_t i0 = w.first; i0 < w.n; i0 += w.step) {
    for (uint32_t e = threadIdx.x; e < kSlots; e += 256u) { key[e] = kNone; cnt[e] = 0u; }
    __syncthreads();
    uint32_t slot[kPer], rank[kPer];
    SegCells c[kPer];
#pragma unroll
    for (uint32_t k = 0; k < kPer; k++) {
      const uint32_t i = i0 + k * 256u + threadIdx.x;
      c[k] = SegCells{kNone, 0u, 0u};
      if (i < w.n) c[k] = seg_cells(s, s.segs[w.base + i], s.seg_cmd[w.base + i]);
    }
#pragma unroll
    for (uint32_t k = 0; k < kPer; k++) {
      slot[k] = kNone;
      rank[k] = 0;
      if (c[k].n > 1u) {
        for (uint32_t b = 0; b < c[k].n; b++) atomicAdd(&s.mat_pres[c[k].cell + (uint64_t)b * c[k].step], 1u);
      }
      else if (c[k].n == 1u) {
        uint32_t h = (c[k].cell * 0x9E3779B1u) >> 23;
        for (uint32_t probe = 0; probe < 8u; probe++, h = (h + 1u) & (kSlots - 1u)) {
          uint32_t have = ((volatile uint32_t*)key)[h];
          if (have == kNone) have = atomicCAS(&key[h], kNone, c[k].cell);
          if (have == kNone || have == c[k].cell) { slot[k] = h; break; }
        }
        // (a full table: straight to the cell)
        rank[k] = slot[k] != kNone ? atomicAdd(&cnt[slot[k]], 1u) : atomicAdd(&s.mat_cnt[c[k].cell], 1u);
      }
    }
    __syncthreads();
    for (uint32_t e = threadIdx.x; e < kSlots; e += 256u)
      if (cnt[e]) at[e] = atomicAdd(&s.mat_cnt[key[e]], cnt[e]);
    __syncthreads();
#pragma unroll
    for (uint32_t k = 0; k < kPer; k++) {
      const uint32_t i = i0 + k * 256u + threadIdx.x;
      if (c[k].n == 1u) s.seg_rank[w.base + i] = rank[k] + (slot[k] != kNone ? at[slot[k]] : 0u);
    }
    __syncthreads();
  }
}

void launch_bin_count(const FrameDev& f, const FrameScratch& s, uint64_t n_segs, hipStream_t st) {
  const uint32_t blocks = f.n_src ? bin_blocks(s, n_segs) : 0u;
  const uint32_t boxes = f.n_boxes ? (uint32_t)(((uint64_t)f.n_cmds * 16 + 255) / 256) : 0u;
  if (!(blocks + boxes)) return;
  if (bin_per(n_segs) == 1) hipLaunchKernelGGL(k_bin_count<1>, dim3(blocks + boxes), dim3(256), 0, st, f, s, blocks);
  else hipLaunchKernelGGL(k_bin_count<kBinPer>, dim3(blocks + boxes), dim3(256), 0, st, f, s, blocks);
}

// Exclusive scans of the (band, command) cells: binned counts and presence
// (a cell with segments, or one a box fill marked) side by side.  Each
// workgroup takes `per` consecutive cells; the first launch sums them, the
// second adds up the sums before its own and scans (one workgroup needs no
// first launch).  The totals go one past the end and to the counters.
constexpr uint32_t kScanMaxBlocks = 2048;
struct ScanPlan { uint32_t blocks; uint64_t per; };
inline ScanPlan scan_plan(uint64_t n, uint64_t min_per) {
  const uint64_t per = std::max<uint64_t>(min_per, ((n + kScanMaxBlocks - 1) / kScanMaxBlocks + 255) / 256 * 256);
  return ScanPlan{(uint32_t)std::max<uint64_t>((n + per - 1) / per, 1), per};
}
size_t scan_tmp_words(void) { return (size_t)kScanMaxBlocks * 4; }

template<int K> struct ScanVal { uint32_t v[K]; };

// Sums of K values over the workgroup (256 threads), and optionally each
// thread's exclusive prefix.
template<int K>
__device__ __forceinline__ ScanVal<K> block_scan(const ScanVal<K>& x, ScanVal<K>* excl) {
  __shared__ uint32_t wsum[K][4];
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
  ScanVal<K> incl, total;
#pragma unroll
  for (int k = 0; k < K; k++) {
    incl.v[k] = lane_scan_add<64>(x.v[k]);
    if (lane == 63) wsum[k][wave] = incl.v[k];
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < K; k++) {
    uint32_t before = 0, all = 0;
#pragma unroll
    for (uint32_t w = 0; w < 4; w++) {
      const uint32_t v = wsum[k][w];
      before += w < wave ? v : 0u;
      all += v;
    }
    total.v[k] = all;
    if (excl) excl->v[k] = before + incl.v[k] - x.v[k];
  }
  __syncthreads();
  return total;
}

template<int K>
__device__ __forceinline__ ScanVal<K> sums_before(const uint32_t* __restrict__ sums) {
  ScanVal<K> x;
#pragma unroll
  for (int k = 0; k < K; k++) x.v[k] = 0u;
  for (uint32_t b = threadIdx.x; b < blockIdx.x; b += 256u)
#pragma unroll
    for (int k = 0; k < K; k++) x.v[k] += sums[(size_t)b * K + k];
  return block_scan<K>(x, nullptr);
}

// Counts and presence of cell i.
__device__ __forceinline__ ScanVal<2> cell_value(const FrameScratch& s, uint64_t i, uint64_t n) {
  ScanVal<2> x{{0u, 0u}};
  if (i < n) {
    const uint32_t mark = s.mat_pres[i];
    x.v[0] = s.mat_cnt[i] + (mark & ~kBoxMark);
    x.v[1] = (x.v[0] | mark) ? 1u : 0u;
  }
  return x;
}

// The class of band b: analytic fills present (a non-empty binned range) ->
// its tiles go to k_render; otherwise its tile groups go to k_render_box_fast
// (solid SRC_OVER / SRC_COPY aligned boxes only), or to k_render_box, the
// solid or the general instance, or, without any command, to none.
__device__ __forceinline__ ScanVal<4> band_value(const FrameDev& f, const FrameScratch& s, uint64_t b, uint64_t n) {
  ScanVal<4> x{{0u, 0u, 0u, 0u}};
  if (b >= n) return x;
  uint32_t lo = 0, hi = f.n_canvases;   // canvas: the last one whose first band is <= b
  while (hi - lo > 1) {
    const uint32_t mid = (lo + hi) >> 1;
    if (f.canvases[mid].band_base <= b) lo = mid; else hi = mid;
  }
  const DevCanvas& cv = f.canvases[lo];
  const uint64_t row_base = cv.mat_base + (b - cv.band_base) * cv.n_cmds;
  const BandClass c = band_class(s.list_off[row_base + cv.n_cmds] - s.list_off[row_base],
                                 s.mat_off[row_base + cv.n_cmds] != s.mat_off[row_base], s.band_nonsolid[b] != 0u, s.band_slow[b] != 0u);
#pragma unroll
  for (uint32_t k = 0; k < 4u; k++) x.v[k] = c == k ? (k == kBandTiles ? cv.tiles_x : cv.groups_x) : 0u;
  return x;
}

template<bool kBands>
__global__ __launch_bounds__(256) void k_scan_sums(FrameDev f, FrameScratch s, uint64_t n, uint64_t per) {
  constexpr int K = kBands ? 4 : 2;
  const uint64_t b0 = (uint64_t)blockIdx.x * per, e = min(b0 + per, n);
  ScanVal<K> x;
#pragma unroll
  for (int k = 0; k < K; k++) x.v[k] = 0u;
  for (uint64_t i = b0 + threadIdx.x; i < e; i += 256u) {
    ScanVal<K> c;
    if constexpr (kBands) c = band_value(f, s, i, e);
    else c = cell_value(s, i, e);
#pragma unroll
    for (int k = 0; k < K; k++) x.v[k] += c.v[k];
  }
  const ScanVal<K> t = block_scan<K>(x, nullptr);
  if (threadIdx.x == 0)
#pragma unroll
    for (int k = 0; k < K; k++) s.scan_tmp[(size_t)blockIdx.x * K + k] = t.v[k];
}

template<bool kBands>
__global__ __launch_bounds__(256) void k_scan_apply(FrameDev f, FrameScratch s, uint64_t n, uint64_t per) {
  constexpr int K = kBands ? 4 : 2;
  uint32_t* out[4] = {s.mat_off, s.list_off, nullptr, nullptr};
  if (kBands) { out[0] = s.tile_off; out[1] = s.fgroup_off; out[2] = s.sgroup_off; out[3] = s.ggroup_off; }
  ScanVal<K> base = sums_before<K>(s.scan_tmp);
  const uint64_t b0 = (uint64_t)blockIdx.x * per, e = min(b0 + per, n);
  for (uint64_t c0 = b0; c0 < e; c0 += 256u) {
    const uint64_t i = c0 + threadIdx.x;
    ScanVal<K> x, excl;
    if constexpr (kBands) x = band_value(f, s, i, e);
    else x = cell_value(s, i, e);
    const ScanVal<K> t = block_scan<K>(x, &excl);
#pragma unroll
    for (int k = 0; k < K; k++) {
      if (i < e) out[k][i] = base.v[k] + excl.v[k];
      base.v[k] += t.v[k];
    }
  }
  if (blockIdx.x + 1 == gridDim.x && threadIdx.x == 0)
#pragma unroll
    for (int k = 0; k < K; k++) {
      out[k][n] = base.v[k];
      s.counters[(kBands ? kCounterTiles : kCounterBinned) + k] = base.v[k];
    }
}

void launch_scans(const FrameDev& f, const FrameScratch& s, hipStream_t st) {
  const ScanPlan c = scan_plan(f.n_mat, 2048);
  if (c.blocks > 1) hipLaunchKernelGGL(k_scan_sums<false>, dim3(c.blocks), dim3(256), 0, st, f, s, f.n_mat, c.per);
  hipLaunchKernelGGL(k_scan_apply<false>, dim3(c.blocks), dim3(256), 0, st, f, s, f.n_mat, c.per);
  const ScanPlan b = scan_plan(f.n_bands, 1024);
  if (b.blocks > 1) hipLaunchKernelGGL(k_scan_sums<true>, dim3(b.blocks), dim3(256), 0, st, f, s, (uint64_t)f.n_bands, b.per);
  hipLaunchKernelGGL(k_scan_apply<true>, dim3(b.blocks), dim3(256), 0, st, f, s, (uint64_t)f.n_bands, b.per);
}

// Copies every segment into its cells: one of a single band to its number's
// place, one that crosses bands to a place behind those, taken from the cell's
// cursor.
template<uint32_t kPer>
__global__ __launch_bounds__(256) void k_bin_scatter(FrameDev f, FrameScratch s) {
  if (pool_overflowed(s)) return;
  // pool mode: the binned pool is sized ahead of time; a larger total is an
  // overflow (the frame falls back to exact counting)
  if (s.binned_cap && s.mat_off[f.n_mat] > s.binned_cap) {
    if (blockIdx.x == 0 && threadIdx.x == 0) atomicOr(s.flags, 2u);
    return;
  }
  const RegionWalk w = region_walk(s, blockIdx.x, gridDim.x, kPer);
  for (uint32_t i0 = w.first; i0 < w.n; i0 += w.step) {
#pragma unroll
    for (uint32_t k = 0; k < kPer; k++) {
      const uint32_t i = i0 + k * 256u + threadIdx.x;
      if (i >= w.n) continue;
      const DevSeg g = s.segs[w.base + i];
      const SegCells c = seg_cells(s, g, s.seg_cmd[w.base + i]);
      if (c.n == 1u) s.binned[s.mat_off[c.cell] + s.seg_rank[w.base + i]] = g;
      else
        for (uint32_t b = 0; b < c.n; b++) s.binned[atomicAdd(&s.mat_pres[c.cell + (uint64_t)b * c.step], 1u)] = g;
    }
  }
}

void launch_bin_scatter(const FrameDev& f, const FrameScratch& s, uint64_t n_segs, hipStream_t st) {
  if (!n_segs || !f.n_src) return;
  const dim3 grid(bin_blocks(s, n_segs));
  if (bin_per(n_segs) == 1) hipLaunchKernelGGL(k_bin_scatter<1>, grid, dim3(256), 0, st, f, s);
  else hipLaunchKernelGGL(k_bin_scatter<kBinPer>, grid, dim3(256), 0, st, f, s);
}

// Command lists of the bands: every present (band, command) cell becomes one
// entry, in command order within its band: the tile-column range (the render
// filter reads only this), {command, binned offset, binned count, what the
// compositor branches on}, and the colour of a solid style or the style index
// of another, so a solid fill needs no command or style record at all.
__device__ __forceinline__ uint32_t cmd_meta(const DevCmd& c, uint32_t fetch_kind) {
  return c.kind | (c.op << kMetaOp) | (c.alpha << kMetaAlpha) | ((c.rule_mask == 0x1FFu ? 1u : 0u) << kMetaEvenOdd) |
         (fetch_kind << kMetaFetch) | (c.src_fmt << kMetaFmt);
}

// Per command, the range of tile columns it can touch, packed as
// first | last << 16 (first > last when it touches none).  Analytic fills
// touch cells min_x .. max_x + 1 of their edges; boxes their pixel box.
__device__ __forceinline__ uint32_t cmd_columns(const FrameScratch& s, const DevCmd& cmd, uint32_t c, const DevCanvas& cv) {
  int x0, x1;
  if (cmd.kind == kCmdAnalytic) {
    const CmdBounds bd = s.bounds[c];
    x0 = bd.min_x;
    x1 = bd.max_x + 1;
  }
  else {
    x0 = cmd.box[0];
    x1 = cmd.box[2] - 1;
  }
  const int last = (int)cv.tiles_x - 1;
  int t0 = x0 < 0 ? 0 : x0 / kTileW;
  int t1 = x1 < 0 ? -1 : x1 / kTileW;
  t1 = t1 > last ? last : t1;
  return (x0 > x1 || t0 > t1) ? 0xFFFFu : ((uint32_t)t0 | ((uint32_t)t1 << 16));
}

__device__ __forceinline__ void list_build(const FrameDev& f, const FrameScratch& s, uint64_t i) {
  const uint32_t li = s.list_off[i], off = s.mat_off[i];
  const bool present = s.list_off[i + 1] != li;
  // the mark is used up: its word becomes the cursor of the segments that
  // cross bands, behind the numbered ones
  s.mat_pres[i] = off + s.mat_cnt[i];
  if (!present) return;
  // canvas of matrix cell i: the last one whose matrix base is <= i
  uint32_t lo = 0, hi = f.n_canvases;
  while (hi - lo > 1) {
    const uint32_t mid = (lo + hi) >> 1;
    if (f.canvases[mid].mat_base <= i) lo = mid; else hi = mid;
  }
  const DevCanvas& cv = f.canvases[lo];
  const uint32_t cmd = cv.cmd_base + (uint32_t)((i - cv.mat_base) % cv.n_cmds);
  const DevCmd& c = f.cmds[cmd];
  const DevStyle& st = f.styles[c.style];
  s.list_cols[li] = cmd_columns(s, c, cmd, cv);
  uint4 ent = make_uint4(cmd, off, s.mat_off[i + 1] - off, cmd_meta(c, st.kind));
  if (c.kind != kCmdAnalytic) {
    const int y0 = (int)((uint32_t)(i - cv.mat_base) / cv.n_cmds) * kTileH;
    ent.y = (uint32_t)c.box[0] | ((uint32_t)c.box[2] << 16);
    ent.z = 0u;
    ent.w |= ((uint32_t)max(c.box[1] - y0, 0) << kMetaRow0) | ((uint32_t)min(c.box[3] - y0, kTileH) << kMetaRow1);
  }
  s.list_ent[li] = ent;
  s.list_style[li] = st.kind == kFetchSolid ? st.solid : c.style;
}

// Compacted headers: {canvas, the band's command list range, column | band
// << 16} for every tile of an analytic band.
__device__ __forceinline__ void tile_setup(const FrameDev& f, const FrameScratch& s, uint32_t i) {
  uint32_t lo = 0, hi = f.n_canvases;
  while (hi - lo > 1) {
    const uint32_t mid = (lo + hi) >> 1;
    if (f.canvases[mid].tile_base <= i) lo = mid; else hi = mid;
  }
  const DevCanvas& cv = f.canvases[lo];
  const uint32_t local = i - cv.tile_base;
  const uint32_t band = local / cv.tiles_x, col = local % cv.tiles_x;
  const uint32_t gb = cv.band_base + band;
  const uint32_t at = s.tile_off[gb];
  if (s.tile_off[gb + 1] == at) return;
  const uint64_t row_base = cv.mat_base + (uint64_t)band * cv.n_cmds;
  s.tile_hdr[at + col] = make_uint4(lo, s.list_off[row_base], s.list_off[row_base + cv.n_cmds], col | (band << 16));
}

// Per box tile group two header words: {canvas, the band's command
// list range, group column | band << 16} and the destination address of the
// group's first pixel {address low, address high, stride, width left of the
// group's first pixel | valid rows << 16 | A8 << 21 | fresh << 22 | tiles << 24},
// so the compositor needs no canvas record.  fresh: the canvas's first command
// copies an opaque colour over the whole group.
__device__ __forceinline__ void group_setup(const FrameDev& f, const FrameScratch& s, uint32_t i) {
  uint32_t lo = 0, hi = f.n_canvases;
  while (hi - lo > 1) {
    const uint32_t mid = (lo + hi) >> 1;
    if (f.canvases[mid].group_base <= i) lo = mid; else hi = mid;
  }
  const DevCanvas& cv = f.canvases[lo];
  const uint32_t local = i - cv.group_base;
  const uint32_t band = local / cv.groups_x, col = local % cv.groups_x;
  const uint32_t gb = cv.band_base + band;
  uint32_t slot;
  if (s.fgroup_off[gb + 1] != s.fgroup_off[gb]) slot = s.fgroup_off[gb] + col;
  else if (s.sgroup_off[gb + 1] != s.sgroup_off[gb]) slot = s.fgroup_off[f.n_bands] + s.sgroup_off[gb] + col;
  else if (s.ggroup_off[gb + 1] != s.ggroup_off[gb]) slot = s.fgroup_off[f.n_bands] + s.sgroup_off[f.n_bands] + s.ggroup_off[gb] + col;
  else return;
  const uint64_t row_base = cv.mat_base + (uint64_t)band * cv.n_cmds;
  const uint32_t tc0 = col * kGroupTiles;
  const uint32_t ntiles = cv.tiles_x - tc0 < (uint32_t)kGroupTiles ? cv.tiles_x - tc0 : (uint32_t)kGroupTiles;
  const uint32_t x0 = tc0 * kTileW, y0 = band * kTileH;
  const uint32_t rows = cv.h - y0 < (uint32_t)kTileH ? cv.h - y0 : (uint32_t)kTileH;
  const uint32_t a8 = cv.format == kFmtA8 ? 1u : 0u;
  const uint64_t ptr = cv.ptr + (uint64_t)((int64_t)y0 * cv.stride) + (uint64_t)x0 * (a8 ? 1u : 4u);
  const uint32_t fresh = starts_opaque(cv, f.cmds, f.styles, x0, y0, min(cv.w, x0 + kGroupTiles * kTileW), y0 + rows) ? 1u : 0u;
  uint4* h = s.group_hdr + 2 * (size_t)slot;
  h[0] = make_uint4(lo, s.list_off[row_base], s.list_off[row_base + cv.n_cmds], col | (band << 16));
  h[1] = make_uint4((uint32_t)ptr, (uint32_t)(ptr >> 32), (uint32_t)cv.stride,
                    min(cv.w - x0, 0xFFFFu) | (rows << 16) | (a8 << 21) | (fresh << 22) | (ntiles << 24));
}

// Lists, scatter cursors and headers in one launch.
__global__ __launch_bounds__(256) void k_setup(FrameDev f, FrameScratch s) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < f.n_mat) list_build(f, s, i);
  if (i < f.n_tiles) tile_setup(f, s, (uint32_t)i);
  if (i < f.n_groups) group_setup(f, s, (uint32_t)i);
}

void launch_setup(const FrameDev& f, const FrameScratch& s, hipStream_t st) {
  const uint64_t n = std::max<uint64_t>(f.n_mat, f.n_tiles);
  if (n) hipLaunchKernelGGL(k_setup, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, f, s);
}

// ---------------------------------------------------------------------------
// Stage 3: render
// ---------------------------------------------------------------------------

// LDS cell buffer of one command in a tile strip: its rows x 64 cells, then
// one backdrop word per row (the summed contributions of cells left of the
// tile).  Within a row the 16 groups of four cells are stored XOR-swizzled by
// the row index, so the same cell column of different rows (the rows of one
// steep edge, rasterized by neighbouring lanes) falls into different LDS
// banks; a group stays four consecutive words, so the compositor still
// reads a thread's four cells with one 128-bit load.
__device__ __forceinline__ int cell_index(int row, int x) {
  return row * kTileW + ((((x >> 2) ^ row) & 15) << 2) + (x & 3);
}

// First pass over one binned segment of an analytic fill, for the rows
// [Y0, Y0 + rows) of a tile: a segment right of the tile is dropped; one left
// of it adds its signed vertical extent per covered row to the backdrop; for
// one that reaches the tile the number of rows it covers is returned, each a
// raster task.
__device__ __forceinline__ uint32_t seg_tile_rows(const DevSeg& g, uint32_t* backdrop, int X0, int Y0, int rows) {
  const int32_t x1 = g.x1 & 0x7FFFFFFF;
  const int32_t cmin = (g.x0 < x1 ? g.x0 : x1) >> 8;
  const int32_t cmax = (g.x0 < x1 ? x1 : g.x0) >> 8;
  int r0 = g.y0 >> 8, r1 = (g.y1 - 1) >> 8;
  if (r0 < Y0) r0 = Y0;
  if (r1 > Y0 + rows - 1) r1 = Y0 + rows - 1;
  if (cmin >= X0 + kTileW || r1 < r0) return 0u;
  if (cmax + 1 < X0) {
    // every cell of every row lies left of the tile: each row adds its y
    // extent, signed by the edge direction (bit 31 of x1)
    const int32_t sgn = g.x1 < 0 ? -1 : 1;
    for (int r = r0; r <= r1; r++) {
      const int lo_y = g.y0 > r * 256 ? g.y0 : r * 256;
      const int hi_y = g.y1 < (r + 1) * 256 ? g.y1 : (r + 1) * 256;
      atomicAdd(&backdrop[r - Y0], (uint32_t)ras::with_sign(hi_y - lo_y, sgn) << 9);
    }
    return 0u;
  }
  return (uint32_t)(r1 - r0 + 1);
}

// Row `r` of a segment that reaches the tile: the closed-form row emitter adds
// the cells inside the tile and one backdrop value for the cells left of it.
__device__ __forceinline__ void raster_row(const DevSeg& g, uint32_t* cells, uint32_t* backdrop, int X0, int Y0, int r) {
  ras::Edge e;
  if (!ras::edge_init(e, g.x0, g.y0, g.x1 & 0x7FFFFFFF, g.y1)) return;
  const int32_t sgn = g.x1 < 0 ? -1 : 1;
  const int lr = r - Y0;
  const uint32_t bd = ras::emit_row(e, r, X0, kTileW, sgn, [&](int32_t k, uint32_t v) {
    if (v) atomicAdd(&cells[cell_index(lr, k)], v);
  });
  if (bd) atomicAdd(&backdrop[lr], bd);
}

// Composited pixels of one wave or workgroup, into one of 64 counters (the
// report sums them).
__device__ __forceinline__ void count_pixels(const FrameScratch& s, unsigned long long n) {
  unsigned long long* px = (unsigned long long*)(s.counters + kCounterPixels);
  if (n) atomicAdd(&px[(blockIdx.x & 63u) * (kPixelStep / 2)], n);
}

// Workgroup -> tile.  Workgroups are dealt to the 8 XCDs round-robin, and an XCD
// takes no work from another, so each gets every eighth run of kXcdRun
// consecutive tiles: a contiguous eighth of the tiles per XCD (better for its
// L2) left the XCDs with the dense parts of a picture working alone.  Render
// stage ms for contiguous eighths / runs of 1 / 4 / 16 / 64: 10 000 cubics
// 1080p 2.77 / 2.06 / 1.98 / 2.01 / 2.14, 2000 pattern shapes 4K 1.41 / 1.21 /
// 1.22 / 1.25 / 1.27, uneven canvases 2.60 / 1.98 / 1.94 / 1.94 / 1.92, 1024
// glyph canvases 1.86 / 1.78 / 1.77 / 1.79 / 1.77, 1000 polygons 512x512 (two
// strips) 0.82 / 0.77 / 0.76 / 0.75 / 0.82.
constexpr uint32_t kXcds = 8, kXcdRun = 4;
// Workgroups that cover n tiles.
inline dim3 xcd_grid(uint32_t n) { return dim3((n + kXcds * kXcdRun - 1) / (kXcds * kXcdRun) * (kXcds * kXcdRun)); }
__device__ __forceinline__ uint32_t xcd_tile(uint32_t wg) {
  const uint32_t at = wg / kXcds;
  return (at / kXcdRun * kXcds + wg % kXcds) * kXcdRun + at % kXcdRun;
}

// Analytic tiles.
//
// What bounds them: instruction issue.  Rasterization is one row of one
// segment per lane, compositing a few dozen integer instructions per pixel and
// command; a tile's destination is read and written once.  So the work is laid
// out for few instructions per command and no waiting on memory in between:
//
//  - everything that belongs to a command is wave-uniform: its list entry
//    arrives in a lane of the wave (63 selected entries at a time) and is read
//    into scalar registers with v_readlane; branches on its kind, operator and
//    style are scalar, other records are scalar loads;
//  - cross-lane sums are DPP moves on the VALU, not LDS permutes;
//  - pixels stay in registers as 16-bit pairs for the packed 16-bit
//    instructions, and a wave with one mask for all its pixels under a solid
//    colour forms the source terms once, in scalar registers;
//  - a wave whose rows a command does not touch skips it after one look at its
//    cells.
//
// Each thread holds N pixels of a row (4, 2 or 1), so a workgroup of four
// waves covers 64 x 4N pixels: a whole 16-row tile, or a half or quarter strip
// of it (see strips_for).
//
// Measured against records in LDS, permute scans and 64-bit divisions per row
// (render stage, one workgroup per tile): 1024 glyph canvases 3.49 -> 1.86 ms
// (VALU instructions 1177 -> 720 million, the VALU three quarters busy),
// 10 000 gradient cubics at 1920x1080 4.60 -> 2.77, 2000 pattern shapes at
// 3840x2160 2.04 -> 1.41, 32 canvases of uneven paths 4.22 -> 2.60, 1000
// polygons at 512x512 2.17 -> 1.01 (0.73 in four strips).
//
// Commands rasterized together.  The segments of a batch's commands are
// spread over all lanes of the workgroup, each command into its own LDS cell
// buffer; after one barrier every wave composites its rows through the
// batch's commands in submission order.  Rasterization of different commands
// is independent, so only the composite has to follow the command order.
constexpr uint32_t kTileBatch = 7;
constexpr uint32_t kTileGroup = 64u / kTileBatch * kTileBatch;   // selected entries held by a wave

// Masks of pixels px .. px + N - 1 of row y for a box fill (uniform command).
template<int N>
__device__ __forceinline__ void box_masks_n(const FrameDev& f, uint4 ent, int y, int px, uint32_t m[N]) {
  const uint32_t kind = ent.w & 3u, alpha = (ent.w >> kMetaAlpha) & 0xFFu;
  const int bx0 = (int)(ent.y & 0xFFFFu), bx1 = (int)(ent.y >> 16);
  const uint32_t row = (uint32_t)y % kTileH;
  const bool row_in = row >= ((ent.w >> kMetaRow0) & 31u) && row < ((ent.w >> kMetaRow1) & 31u);
  if (kind == kCmdBoxA) {
#pragma unroll
    for (int k = 0; k < N; k++) m[k] = (row_in && px + k >= bx0 && px + k < bx1) ? alpha : 0u;
    return;
  }
  const pipe::CPtr<DevCmd> c = pipe::cptr(f.cmds + ent.x);
  if (kind == kCmdBoxM) {
    // FillMask with a VMaskA8 command (rendercommandprocsync_p.h:65-84,
    // compopgeneric_p.h:165-183): byte x - x0 of the mask row, times the
    // alpha below full alpha.  The view is exactly the box (host-checked), so
    // every byte read lies in row y - y0 of the view.
    const pipe::CPtr<DevImage> mi = pipe::cptr(f.images + c->box_mask[0]);
    const pipe::GBytes bytes = pipe::global_bytes(mi->ptr) + (int64_t)(y - c->box[1]) * mi->stride - bx0;
    if (N == 4 && row_in && px >= bx0 && px + 3 < bx1) {
      typedef uint32_t bytes4 __attribute__((aligned(1)));
      const uint32_t v = *(const B2AMD_GLOBAL bytes4*)(bytes + px);
#pragma unroll
      for (int k = 0; k < N; k++) m[k] = (v >> (8 * k)) & 0xFFu;
    }
    else {
#pragma unroll
      for (int k = 0; k < N; k++) {
        m[k] = 0u;
        if (row_in && px + k >= bx0 && px + k < bx1) m[k] = bytes[px + k];
      }
    }
    if (alpha < 255u) {
#pragma unroll
      for (int k = 0; k < N; k++) m[k] = pipe::div255(m[k] * alpha);
    }
  }
  else {
    const uint32_t top = c->box_mask[0], mid = c->box_mask[1], bot = c->box_mask[2];
    const uint32_t rm = y == c->box_row_first ? top : y == c->box_row_last ? bot : mid;
#pragma unroll
    for (int k = 0; k < N; k++) {
      const int x = px + k;
      const uint32_t sh = x == bx0 ? 0u : x == bx1 - 1 ? 16u : 8u;
      m[k] = (row_in && x >= bx0 && x < bx1) ? (rm >> sh) & 0xFFu : 0u;
    }
  }
}

// Masks of four pixels from px on in each of R rows from y on (uniform), one
// byte each, for a box that isn't kCmdBoxA.  All rows' bytes are loaded before
// any is used.
template<int R>
__device__ __forceinline__ void box_mask_rows(const FrameDev& f, uint4 ent, int y, int px, uint32_t pm[R]) {
  const uint32_t alpha = (ent.w >> kMetaAlpha) & 0xFFu;
  const int bx0 = (int)(ent.y & 0xFFFFu), bx1 = (int)(ent.y >> 16);
  const pipe::CPtr<DevCmd> c = pipe::cptr(f.cmds + ent.x);
  const int by0 = c->box[1], by1 = c->box[3];
#pragma unroll
  for (int r = 0; r < R; r++) pm[r] = 0u;
  if ((ent.w & 3u) == kCmdBoxM) {
    // see box_masks_n; rows outside the box read its nearest one and drop it
    const pipe::CPtr<DevImage> mi = pipe::cptr(f.images + c->box_mask[0]);
    const pipe::GBytes at = pipe::global_bytes(mi->ptr) - bx0;
    const int64_t stride = mi->stride;
    auto row = [&](int r) { return at + (int64_t)(min(max(y + r, by0), by1 - 1) - by0) * stride; };
    if (px >= bx0 && px + 3 < bx1) {
      typedef uint32_t bytes4 __attribute__((aligned(1)));
#pragma unroll
      for (int r = 0; r < R; r++) pm[r] = *(const B2AMD_GLOBAL bytes4*)(row(r) + px);
    }
    else if (px < bx1 && px + 3 >= bx0) {
#pragma unroll
      for (int k = 0; k < 4; k++) {
        if (px + k < bx0 || px + k >= bx1) continue;
#pragma unroll
        for (int r = 0; r < R; r++) pm[r] |= (uint32_t)row(r)[px + k] << (8 * k);
      }
    }
    if (alpha < 255u) {
#pragma unroll
      for (int r = 0; r < R; r++) {
        const pipe::Px p = pipe::px_of(pm[r]);
        pm[r] = pipe::px_bits(pipe::Px{pipe::div255p(p.rb * (uint16_t)alpha), pipe::div255p(p.ag * (uint16_t)alpha)});
      }
    }
  }
  else {
    const uint32_t top = c->box_mask[0], mid = c->box_mask[1], bot = c->box_mask[2];
    const int first = c->box_row_first, last = c->box_row_last;
    uint32_t sh[4];
    bool in[4];
#pragma unroll
    for (int k = 0; k < 4; k++) {
      const int x = px + k;
      sh[k] = x == bx0 ? 0u : x == bx1 - 1 ? 16u : 8u;
      in[k] = x >= bx0 && x < bx1;
    }
#pragma unroll
    for (int r = 0; r < R; r++) {
      const uint32_t rm = y + r == first ? top : y + r == last ? bot : mid;
#pragma unroll
      for (int k = 0; k < 4; k++) pm[r] |= in[k] ? ((rm >> sh[k]) & 0xFFu) << (8 * k) : 0u;
    }
  }
#pragma unroll
  for (int r = 0; r < R; r++)
    if (y + r < by0 || y + r >= by1) pm[r] = 0u;
}

// A solid colour over the whole wave under one mask (32-bit SRC_OVER and
// SRC_COPY): composited with the source terms formed once; false otherwise.
template<int N>
__device__ __forceinline__ bool solid_flat(uint32_t op, uint32_t color, const uint32_t m[N], pipe::Px d[N]) {
  if (op > kOpSrcOver) return false;
  const uint32_t m0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)m[0]);
  uint32_t diff = m[0] ^ m0;
#pragma unroll
  for (int k = 1; k < N; k++) diff |= m[k] ^ m0;
  if (__ballot(diff != 0u)) return false;
  pipe::composite32_flat<N>(op, d, color, m0);
  return true;
}

// One command's pixels: fetch and composite under masks m.
template<int N, bool kDither>
__device__ __forceinline__ void apply_n(const FrameDev& f, const FrameScratch& s, uint32_t meta, uint32_t cmd, uint32_t style,
                                        bool a8, uint32_t ref_band_h, int y, int px, const uint32_t m[N], pipe::Px d[N]) {
  const uint32_t op = (meta >> kMetaOp) & 7u, fetch = (meta >> kMetaFetch) & 7u;
  constexpr int kPairs = (N + 1) / 2;
  uint32_t src[N];
  if (fetch == kFetchSolid) {
    if (!a8 && solid_flat<N>(op, style, m, d)) return;
#pragma unroll
    for (int k = 0; k < N; k++) src[k] = style;
  }
  else {
    uint32_t any = m[0];
#pragma unroll
    for (int k = 1; k < N; k++) any |= m[k];
#pragma unroll
    for (int k = 0; k < N; k++) src[k] = 0u;
    if (any) {
      int row0 = 0;
      const bool analytic = (meta & 3u) == kCmdAnalytic;
      if (fetch == kFetchConic) row0 = analytic ? pipe::cptr(s.bounds + cmd)->min_y >> 8 : (int)pipe::cptr(f.cmds + cmd)->fetch_row0;
      pipe::fetch_n<N, kDither>(pipe::cptr(f.styles + style), fetch, y, px, row0, analytic ? ref_band_h : 0u, f.luts, f.images,
                                (meta >> kMetaFmt) & 3u, src);
    }
  }
  if (a8) {
    pipe::u16x2 da[kPairs], sa[kPairs], ma[kPairs];
#pragma unroll
    for (int k = 0; k < kPairs; k++) {
      da[k] = d[k].rb;
      const uint32_t k1 = 2 * k + 1 < N ? 2 * k + 1 : 2 * k;
      sa[k] = pipe::u16x2{(uint16_t)(src[2 * k] >> 24), (uint16_t)(src[k1] >> 24)};
      ma[k] = pipe::u16x2{(uint16_t)m[2 * k], (uint16_t)m[k1]};
    }
    pipe::composite8_n<kPairs>(op, da, sa, ma);
#pragma unroll
    for (int k = 0; k < kPairs; k++) d[k].rb = da[k];
    return;
  }
  pipe::Px sp[N];
  pipe::u16x2 mm[N];
#pragma unroll
  for (int k = 0; k < N; k++) {
    sp[k] = pipe::px_of(src[k]);
    mm[k] = pipe::both(m[k]);
  }
  pipe::composite32_n<N>(op, d, sp, mm, fetch >= kFetchPatternNN);
}

// Words px .. px + N - 1 of a row; those past its end stay as they are.
template<int N>
__device__ __forceinline__ void load_words(const uint8_t* rowp, int px, int w, uint32_t v[N]) {
  const uint32_t* r32 = (const uint32_t*)rowp;
  if (N == 4 && px + 3 < w && (((uintptr_t)(r32 + px)) & 15) == 0) {
    const uint4 q = *(const uint4*)(r32 + px);
    const uint32_t u[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
    for (int k = 0; k < N; k++) v[k] = u[k];
  }
  else {
#pragma unroll
    for (int k = 0; k < N; k++) if (px + k < w) v[k] = r32[px + k];
  }
}

template<int N, bool kStream>
__device__ __forceinline__ void store_words(uint8_t* rowp, int px, int w, const uint32_t v[N]) {
  uint32_t* r32 = (uint32_t*)rowp;
  if (N == 4 && px + 3 < w && (((uintptr_t)(r32 + px)) & 15) == 0) {
    typedef uint32_t words4 __attribute__((ext_vector_type(4)));
    const words4 q = {v[0], v[1 % N], v[2 % N], v[3 % N]};
    if (kStream) __builtin_nontemporal_store(q, (words4*)(r32 + px));
    else *(words4*)(r32 + px) = q;
  }
  else {
#pragma unroll
    for (int k = 0; k < N; k++) if (px + k < w) r32[px + k] = v[k];
  }
}

// Destination pixels px .. px + N - 1 of a row, as pairs (A8: neighbouring
// pixels in d[k].rb); zero outside the canvas.
template<int N>
__device__ __forceinline__ void load_px(const uint8_t* rowp, int px, int w, bool a8, pipe::Px d[N]) {
  uint32_t v[N];
#pragma unroll
  for (int k = 0; k < N; k++) v[k] = 0u;
  if (a8) {
    if (N == 4 && px + 3 < w && (((uintptr_t)(rowp + px)) & 3) == 0) {
      const uint32_t b = *(const uint32_t*)(rowp + px);
#pragma unroll
      for (int k = 0; k < N; k++) v[k] = (b >> (8 * k)) & 0xFFu;
    }
    else {
#pragma unroll
      for (int k = 0; k < N; k++) if (px + k < w) v[k] = rowp[px + k];
    }
#pragma unroll
    for (int k = 0; k < (N + 1) / 2; k++) d[k].rb = pipe::u16x2{(uint16_t)v[2 * k], (uint16_t)(2 * k + 1 < N ? v[2 * k + 1 < N ? 2 * k + 1 : 0] : 0u)};
    return;
  }
  load_words<N>(rowp, px, w, v);
#pragma unroll
  for (int k = 0; k < N; k++) d[k] = pipe::px_of(v[k]);
}

template<int N, bool kStream = false>
__device__ __forceinline__ void store_px(uint8_t* rowp, int px, int w, bool a8, const pipe::Px d[N]) {
  if (a8) {
    uint32_t v[N];
#pragma unroll
    for (int k = 0; k < N; k++) v[k] = (pipe::as_u32(d[k / 2].rb) >> (16 * (k & 1))) & 0xFFu;
    if (N == 4 && px + 3 < w && (((uintptr_t)(rowp + px)) & 3) == 0) {
      uint32_t b = 0;
#pragma unroll
      for (int k = 0; k < N; k++) b |= v[k] << (8 * k);
      *(uint32_t*)(rowp + px) = b;
    }
    else {
#pragma unroll
      for (int k = 0; k < N; k++) if (px + k < w) rowp[px + k] = (uint8_t)v[k];
    }
    return;
  }
  uint32_t v[N];
#pragma unroll
  for (int k = 0; k < N; k++) v[k] = pipe::px_bits(d[k]);
  store_words<N, kStream>(rowp, px, w, v);
}

// Rows strip * 4N .. + 4N - 1 of the analytic tile with header `slot`: the
// whole workgroup rasterizes the band's commands that reach the tile and
// composites them in order.  Returns the pixels that this wave composited.
template<int N, bool kDither>
__device__ __forceinline__ uint32_t render_tile(const FrameDev& f, const FrameScratch& s, uint32_t slot, uint32_t strip) {
  constexpr int kRows = 4 * N, kLanes = kTileW / N;   // rows of the strip, lanes per row
  constexpr int kCells = kRows * kTileW, kCellWords = kCells + kRows;
  constexpr uint32_t kB = kTileBatch;
  __shared__ __align__(16) uint32_t cells[kB][kCellWords];
  // Row tasks, per wave: the segments that reach the strip, each with its
  // first task index and batch slot, and the owners of the next 64 tasks.
  __shared__ DevSeg task_seg[kTileThreads / 64][64];
  __shared__ uint32_t task_meta[kTileThreads / 64][64];
  __shared__ uint32_t task_own[kTileThreads / 64][64];
  __shared__ uint8_t sel[kTileThreads];
  __shared__ uint32_t sel_wave[kTileThreads / 64];
  const int t = threadIdx.x;
  const int lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const uint32_t* const hdr = (const uint32_t*)(s.tile_hdr + slot);
  const pipe::CPtr<uint32_t> th = pipe::cptr(hdr);
  const pipe::CPtr<DevCanvas> cv = pipe::cptr(f.canvases + th[0]);
  const uint32_t lb = th[1], le = th[2];
  const uint32_t tcol = th[3] & 0xFFFFu, band = th[3] >> 16;
  // A pool overflow leaves the frame incomplete: nothing is composited and
  // the host redoes the frame with exact counting.
  if (s.flags && *s.flags) return 0;
  const int X0 = (int)tcol * kTileW;
  const int Y0 = (int)band * kTileH + (int)strip * kRows;
  const int w = (int)cv->w;
  const bool a8 = cv->format == kFmtA8;
  const uint32_t ref_band_h = cv->ref_band_h;

  const int row = wave * N + lane / kLanes;   // within the strip
  const int q = lane % kLanes;
  const int y = Y0 + row;
  const int px = X0 + q * N;
  const bool row_ok = y < (int)cv->h;
  // Lanes whose pixel k lies inside the canvas.  The others are composited
  // like any (every fetch is safe at any position) but not counted or stored.
  uint64_t inside[N];
#pragma unroll
  for (int k = 0; k < N; k++) inside[k] = __ballot(row_ok && px + k < w);

  // zero LDS (each thread its own swizzled group of cells)
  const int grp = cell_index(row, q * N);
#pragma unroll
  for (uint32_t b = 0; b < kB; b++) {
#pragma unroll
    for (int k = 0; k < N; k++) cells[b][grp + k] = 0u;
    if (q == 0) cells[b][kCells + row] = 0u;
  }

  // load the destination pixels
  pipe::Px d[N];
#pragma unroll
  for (int k = 0; k < N; k++) d[k] = pipe::px_of(0u);
  uint8_t* const rowp = (uint8_t*)cv->ptr + (int64_t)y * cv->stride;
  if (row_ok) load_px<N>(rowp, px, w, a8, d);

  // Batch segment index of this thread in the first 256 of a batch: the
  // batch's segments are dealt to the four waves in turn, so every SIMD of
  // the CU takes part in rasterization.
  const uint32_t jt = ((uint32_t)lane << 2) | (uint32_t)wave;
  bool touched = false;
  uint32_t npix = 0;   // composited pixels of the wave

  // The band's command list is filtered 256 entries at a time down to the
  // commands whose tile-column range holds this tile (ballot compaction,
  // submission order kept).
  for (uint32_t chunk = lb; chunk < le; chunk += kTileThreads) {
    const uint32_t li = chunk + (uint32_t)t;
    bool keep = false;
    if (li < le) {
      const uint32_t cols = s.list_cols[li];
      keep = tcol >= (cols & 0xFFFFu) && tcol <= (cols >> 16);
    }
    const uint64_t bal = __ballot(keep);
    if (lane == 0) sel_wave[wave] = (uint32_t)__popcll(bal);
    __syncthreads();   // also: the previous chunk's selection is consumed
    uint32_t off = 0, n_sel = 0;
#pragma unroll
    for (int v = 0; v < kTileThreads / 64; v++) {
      const uint32_t cw = sel_wave[v];
      off += v < wave ? cw : 0u;
      n_sel += cw;
    }
    if (keep) sel[off + (uint32_t)__popcll(bal & ((1ull << lane) - 1ull))] = (uint8_t)t;
    __syncthreads();
    n_sel = (uint32_t)__builtin_amdgcn_readfirstlane((int)n_sel);

    for (uint32_t g0 = 0; g0 < n_sel; g0 += kTileGroup) {
      // up to kTileGroup selected entries, one per lane
      const uint32_t gn = min(n_sel - g0, kTileGroup);
      uint4 ent = make_uint4(0u, 0u, 0u, 0u);
      uint32_t style = 0;
      if ((uint32_t)lane < gn) {
        const uint32_t i = chunk + sel[g0 + (uint32_t)lane];
        ent = s.list_ent[i];
        style = s.list_style[i];
      }
      const uint32_t incl = lane_scan_add<64>(ent.z);      // segments up to and with this entry
      const uint32_t delta = ent.y - (incl - ent.z);       // binned index of group segment j: delta + j

      // the batch's segment `j` (of `total`, the first being group segment
      // `base`): its batch slot and record
      auto find = [&](uint32_t kb, uint32_t nb, uint32_t base, uint32_t j, DevSeg& g) -> uint32_t {
        uint32_t b = 0;
#pragma unroll
        for (uint32_t i = 0; i + 1 < kB; i++) {
          const uint32_t end = i + 1 < nb ? lane_value(incl, kb + i) - base : 0xFFFFFFFFu;
          b += j >= end ? 1u : 0u;
        }
        const uint32_t at = (uint32_t)__shfl((int)delta, (int)(kb + b), 64) + base + j;
        g = s.binned[at];
        return b;
      };
      // (every lane calls it, so the shuffle sees all lanes; lanes past the
      // batch's segments look at its first one and drop it)
      auto batch_n = [&](uint32_t kb) { return min(gn - kb, kB); };
      auto batch_base = [&](uint32_t kb) { return kb ? lane_value(incl, kb - 1u) : 0u; };
      auto batch_total = [&](uint32_t kb) { return lane_value(incl, kb + batch_n(kb) - 1u) - batch_base(kb); };
      DevSeg pre{0, 0, 0, 0};
      uint32_t pre_b = 0;
      uint32_t total = batch_total(0);
      if (total) pre_b = find(0, batch_n(0), 0u, jt < total ? jt : 0u, pre);

      for (uint32_t kb = 0; kb < gn; kb += kB) {
        const uint32_t nb = batch_n(kb), base = batch_base(kb);
        const uint32_t tot = total;
        const DevSeg seg = pre;
        const uint32_t seg_b = pre_b;
        // the next batch's first segments are on their way while this batch
        // is rasterized and composited
        if (kb + kB < gn) {
          total = batch_total(kb + kB);
          if (total) pre_b = find(kb + kB, batch_n(kb + kB), batch_base(kb + kB), jt < total ? jt : 0u, pre);
        }

        // Rasterize the batch.  Segments left of the tile add their row
        // covers to the backdrop; every segment that reaches the strip
        // becomes one task per row it covers, so a lane's serial cell walk
        // is one row long.  A wave's tasks are its own segments': no barrier.
        for (uint32_t rb = 0; rb < tot; rb += kTileThreads) {
          const uint32_t j = rb + jt;
          DevSeg g = seg;
          uint32_t gb = seg_b;
          if (rb) gb = find(kb, nb, base, j < tot ? j : 0u, g);
          const uint32_t rows = j < tot ? seg_tile_rows(g, &cells[gb][kCells], X0, Y0, kRows) : 0u;
          const uint32_t tend = lane_scan_add<64>(rows);
          const uint32_t n_tasks = lane_value(tend, 63u);
          if (n_tasks == 0) continue;
          const uint32_t first = tend - rows;
          if (rows) {
            task_seg[wave][lane] = g;
            task_meta[wave][lane] = first | (gb << 16);
          }
          uint32_t carry = 0;   // owner of the task before this window, + 1
          for (uint32_t k0 = 0; k0 < n_tasks; k0 += 64) {
            // owner of each task of the window: the last segment whose first
            // task is at or before it
            task_own[wave][lane] = 0u;
            wave_sync();
            if (rows && first - k0 < 64u) task_own[wave][first - k0] = (uint32_t)lane + 1u;
            wave_sync();
            const uint32_t own = max(wave_scan_max(task_own[wave][lane]), carry);
            carry = lane_value(own, 63u);
            const uint32_t k = k0 + (uint32_t)lane;
            if (k < n_tasks) {
              const uint32_t o = own - 1u;
              const DevSeg og = task_seg[wave][o];
              const uint32_t tm = task_meta[wave][o];
              const int r0 = (og.y0 >> 8) > Y0 ? (og.y0 >> 8) : Y0;
              uint32_t* cb = cells[tm >> 16];
              raster_row(og, cb, cb + kCells, X0, Y0, r0 + (int)(k - (tm & 0xFFFFu)));
            }
            wave_sync();
          }
        }
        if (tot) __syncthreads();   // cells complete

        // composite the batch's commands in order
        for (uint32_t b = 0; b < nb; b++) {
          const uint32_t p = kb + b;
          const uint32_t meta = lane_value(ent.w, p);
          const uint32_t alpha = (meta >> kMetaAlpha) & 0xFFu;
          uint32_t m[N];
          if ((meta & 3u) == kCmdAnalytic) {
            if (lane_value(ent.z, p) == 0u) continue;
            uint32_t* cb = cells[b];
            uint32_t c[N];
#pragma unroll
            for (int k = 0; k < N; k++) c[k] = cb[grp + k];
            const uint32_t bd = cb[kCells + row];
            uint32_t any = c[0];
#pragma unroll
            for (int k = 1; k < N; k++) any |= c[k];
            const uint64_t has = __ballot(any != 0u);
            if ((has | __ballot(bd != 0u)) == 0ull) continue;   // nothing covers the wave's rows
            uint32_t cov = bd;
            if (has) {
              uint32_t sum = c[0];
#pragma unroll
              for (int k = 1; k < N; k++) sum += c[k];
              cov += lane_scan_add<kLanes>(sum) - sum;
#pragma unroll
              for (int k = 0; k < N; k++) cb[grp + k] = 0u;
            }
            if (q == 0) cb[kCells + row] = 0u;
            // coverage (cov / 512, rounded down) to mask: its magnitude up
            // to 256, folded into [0, 256] first under the even-odd rule
            if ((meta >> kMetaEvenOdd) & 1u) {
#pragma unroll
              for (int k = 0; k < N; k++) {
                cov += c[k];
                const int32_t v = (((int32_t)cov >> 9) + 256 & 0x1FF) - 256;
                m[k] = __umul24((uint32_t)(v < 0 ? -v : v), alpha) >> 8;
              }
            }
            else {
#pragma unroll
              for (int k = 0; k < N; k++) {
                cov += c[k];
                const int32_t v = (int32_t)cov >> 9;
                m[k] = __umul24(min((uint32_t)max(v, -v), 256u), alpha) >> 8;
              }
            }
          }
          else {
            box_masks_n<N>(f, make_uint4(lane_value(ent.x, p), lane_value(ent.y, p), 0u, meta), y, px, m);
          }
          uint32_t n = 0;
#pragma unroll
          for (int k = 0; k < N; k++) n += (uint32_t)__popcll(__ballot(m[k] != 0u) & inside[k]);
          if (n == 0) continue;
          npix += n;
          touched = true;
          apply_n<N, kDither>(f, s, meta, lane_value(ent.x, p), lane_value(style, p), a8, ref_band_h, y, px, m, d);
        }
        if (tot) __syncthreads();   // cells cleared
      }
    }
  }

  if (lane == 0) count_pixels(s, npix);
  if (touched && row_ok) store_px<N>(rowp, px, w, a8, d);
  return npix;
}

// Four workgroups per CU: LDS (7 cell buffers) and the register budget are
// sized for it.  One workgroup per analytic tile or strip.
template<int N, bool kDither>
__global__ __launch_bounds__(kTileThreads, 4) void k_render(FrameDev f, FrameScratch s, uint32_t n) {
  constexpr uint32_t kStrips = 4 / N;
  const uint32_t unit = xcd_tile(blockIdx.x);
  const uint32_t slot = unit / kStrips;
  // uniform: padding workgroups of the XCD mapping, and (when n is an upper
  // bound) slots past the analytic tiles
  if (slot >= n || slot >= s.tile_off[f.n_bands]) return;
  render_tile<N, kDither>(f, s, slot, unit % kStrips);
}

// The same tiles drained from a work queue by a persistent grid: every
// workgroup takes the next queue position with one atomic until the queue is
// exhausted (every workgroup reaches that exit).  The queue holds the
// analytic tile slots in the order k_tile_scatter wrote (longest predicted
// first), or is the identity (null: band order).  With `s.tile_cycles` set
// (2 x the tile count), the wall-clock ticks (100 MHz) of every tile and
// then its composited pixels are logged (cost-model samples).
template<bool kLog, int kOcc, bool kDither>
__global__ __launch_bounds__(kTileThreads, kOcc) void k_render_queue(FrameDev f, FrameScratch s) {
  __shared__ uint32_t next;
  const uint32_t total = s.tile_off[f.n_bands];
  for (;;) {
    __syncthreads();   // the previous tile's LDS reads are done and `next` is free
    if (threadIdx.x == 0) next = atomicAdd(s.queue_head, 1u);
    __syncthreads();
    const uint32_t i = next;
    if (i >= total) break;   // uniform
    const uint32_t slot = s.queue ? s.queue[i] : i;
    if constexpr (!kLog) {
      render_tile<4, kDither>(f, s, slot, 0);
    }
    else {
      __shared__ uint32_t tile_px;
      if (threadIdx.x == 0) tile_px = 0u;
      const long long c0 = wall_clock64();
      const uint32_t px = render_tile<4, kDither>(f, s, slot, 0);
      if ((threadIdx.x & 63u) == 0) atomicAdd(&tile_px, px);
      __syncthreads();
      if (threadIdx.x == 0) {
        s.tile_cycles[slot] = (uint32_t)min((long long)0xFFFFFFFF, wall_clock64() - c0);
        s.tile_cycles[total + slot] = tile_px;
      }
    }
  }
}

// ---------------------------------------------------------------------------
// Work queue of the analytic tiles
// ---------------------------------------------------------------------------

// Per analytic tile the 16 features of the tile cost model, from one walk of
// the band's command list by one wave (the list entries whose tile-column
// range holds the tile are the commands the tile composites):
//   0 log2(1 + commands)          1 log2(1 + binned segments of them)
//   2 log2(1 + segments of commands starting left of the tile)
//   3 log2(1 + list entries of the band)
//   4..8 log2(1 + commands by style: linear, radial, conic, pattern, solid)
//   9 log2(1 + box commands)      10 log2(1 + commands not SRC_OVER)
//   11 A8 canvas                  12 valid rows / 16   13 valid columns / 64
//   14 log2(1 + command batches)  15 log2(1 + largest segment count of one command)
__global__ __launch_bounds__(256) void k_tile_features(FrameDev f, FrameScratch s, uint32_t n) {
  const uint32_t slot = blockIdx.x * 4 + (threadIdx.x >> 6);
  const uint32_t lane = threadIdx.x & 63;
  if (slot >= n || slot >= s.tile_off[f.n_bands]) return;   // uniform per wave
  const uint4 th = s.tile_hdr[slot];
  const DevCanvas& cv = f.canvases[th.x];
  const uint32_t tcol = th.w & 0xFFFFu, band = th.w >> 16;
  uint32_t c[12] = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};   // n, segs, segs_left, lin, rad, con, pat, solid, box, op, -, max
  for (uint32_t li = th.y + lane; li < th.z; li += 64) {
    const uint32_t cols = s.list_cols[li];
    const uint32_t lo = cols & 0xFFFFu, hi = cols >> 16;
    if (tcol < lo || tcol > hi) continue;
    const uint4 ent = s.list_ent[li];
    const uint32_t kind = (ent.w >> kMetaFetch) & 7u;
    c[0] += 1u;
    c[1] += ent.z;
    c[2] += lo < tcol ? ent.z : 0u;
    c[3] += kind == kFetchLinear;
    c[4] += kind == kFetchRadial;
    c[5] += kind == kFetchConic;
    c[6] += kind >= kFetchPatternNN;
    c[7] += kind == kFetchSolid;
    c[8] += (ent.w & 3u) != kCmdAnalytic;
    c[9] += ((ent.w >> kMetaOp) & 7u) != kOpSrcOver;
    c[11] = ent.z > c[11] ? ent.z : c[11];
  }
#pragma unroll
  for (int k = 0; k < 12; k++) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      const uint32_t v = __shfl_xor(c[k], o, 64);
      c[k] = k == 11 ? (v > c[k] ? v : c[k]) : c[k] + v;
    }
  }
  if (lane != 0) return;
  const uint32_t x0 = tcol * kTileW, y0 = band * kTileH;
  const uint32_t rows = cv.h - y0 < (uint32_t)kTileH ? cv.h - y0 : (uint32_t)kTileH;
  const uint32_t cols = cv.w - x0 < (uint32_t)kTileW ? cv.w - x0 : (uint32_t)kTileW;
  float* o = s.tile_feat + (size_t)slot * 16;
  o[0] = log2f(1.0f + (float)c[0]);
  o[1] = log2f(1.0f + (float)c[1]);
  o[2] = log2f(1.0f + (float)c[2]);
  o[3] = log2f(1.0f + (float)(th.z - th.y));
#pragma unroll
  for (int k = 0; k < 5; k++) o[4 + k] = log2f(1.0f + (float)c[3 + k]);
  o[9] = log2f(1.0f + (float)c[8]);
  o[10] = log2f(1.0f + (float)c[9]);
  o[11] = cv.format == kFmtA8 ? 1.0f : 0.0f;
  o[12] = (float)rows / (float)kTileH;
  o[13] = (float)cols / (float)kTileW;
  o[14] = log2f(1.0f + (float)((c[0] + kTileBatch - 1) / kTileBatch));
  o[15] = log2f(1.0f + (float)c[11]);
}

// Queue key of each analytic tile: its predicted cost (log2 ticks from the
// model's first output when `pred` is set, else log2 of binned segments +
// 16 x commands from the features) in 1/8 steps, as a bucket of a
// descending counting sort; bucket sizes into `hist` (256 entries, zeroed),
// counted per workgroup in LDS first (most tiles of a frame fall into a few
// buckets, so per-tile global atomics would queue on them).
constexpr uint32_t kQueueBuckets = 256;
__global__ __launch_bounds__(kQueueBuckets) void k_tile_keys(FrameDev f, FrameScratch s, uint32_t n, const float* __restrict__ pred) {
  __shared__ uint32_t lhist[kQueueBuckets];
  lhist[threadIdx.x] = 0u;
  __syncthreads();
  const uint32_t slot = blockIdx.x * blockDim.x + threadIdx.x;
  if (slot < n && slot < s.tile_off[f.n_bands]) {
    float cost;
    if (pred) {
      cost = pred[(size_t)slot * 2];
    }
    else {
      const float* x = s.tile_feat + (size_t)slot * 16;
      cost = log2f(1.0f + (exp2f(x[1]) - 1.0f) + 16.0f * (exp2f(x[0]) - 1.0f));
    }
    float q = cost * 8.0f;
    q = q != q ? 0.0f : q;   // a NaN prediction sorts last
    const uint32_t key = q <= 0.0f ? 0u : q >= (float)(kQueueBuckets - 1) ? kQueueBuckets - 1 : (uint32_t)q;
    const uint32_t bucket = kQueueBuckets - 1 - key;
    s.tile_key[slot] = bucket;
    atomicAdd(&lhist[bucket], 1u);
  }
  __syncthreads();
  if (lhist[threadIdx.x]) atomicAdd(&s.queue_hist[threadIdx.x], lhist[threadIdx.x]);
}

// Exclusive scan of the bucket sizes in place (one workgroup), and the queue
// head reset.
__global__ __launch_bounds__(kQueueBuckets) void k_queue_scan(FrameScratch s) {
  __shared__ uint32_t v[kQueueBuckets];
  const uint32_t t = threadIdx.x;
  v[t] = s.queue_hist[t];
  __syncthreads();
  for (uint32_t d = 1; d < kQueueBuckets; d <<= 1) {
    const uint32_t a = t >= d ? v[t - d] : 0u;
    __syncthreads();
    v[t] += a;
    __syncthreads();
  }
  s.queue_hist[t] = v[t] - s.queue_hist[t];
  if (t == 0) *s.queue_head = 0u;
}

// Queue positions: each workgroup takes one range per bucket from the
// bucket cursors and numbers its tiles within it in LDS (within a bucket
// the order is any: tiles are independent).
__global__ __launch_bounds__(kQueueBuckets) void k_tile_scatter(FrameDev f, FrameScratch s, uint32_t n) {
  __shared__ uint32_t lcount[kQueueBuckets], lbase[kQueueBuckets];
  lcount[threadIdx.x] = 0u;
  __syncthreads();
  const uint32_t slot = blockIdx.x * blockDim.x + threadIdx.x;
  const bool on = slot < n && slot < s.tile_off[f.n_bands];
  uint32_t bucket = 0, rank = 0;
  if (on) {
    bucket = s.tile_key[slot];
    rank = atomicAdd(&lcount[bucket], 1u);
  }
  __syncthreads();
  if (lcount[threadIdx.x]) lbase[threadIdx.x] = atomicAdd(&s.queue_hist[threadIdx.x], lcount[threadIdx.x]);
  __syncthreads();
  if (on) s.queue[lbase[bucket] + rank] = slot;
}

// Bands with box fills only: one workgroup per group of up to 4 tiles of a
// band (256 x 16 pixels).  What bounds them is memory: every destination pixel
// read and written once, a blit's or mask's pixels read once.  So wave w takes
// rows 4w .. 4w + 3 and lane l the pixels 4l .. 4l + 3 of each: every load and
// store of a wave moves one contiguous 1 KB row segment, those of four rows are
// in flight together, and no LDS or barrier keeps waves from filling the CU.
// The band's commands (kind, colour and box of 64 at a time) sit in the lanes
// of the wave and are read into scalar registers, so that all branches are
// scalar; a command's own fields are read once for the four rows.  Where the
// canvas's first command is an opaque colour over the whole group the
// destination isn't read at all.
//
// Kernels: solid SRC_OVER / SRC_COPY aligned boxes on 32-bit canvases (one of
// its own, k_render_box_fast), other solid styles, and every style.  Measured
// against one thread per 16 pixels of a row with records in LDS, 4K canvases:
// four with an image, a half-size one at a fraction or scaled and 24 sprites
// 422 -> 119 us, two with a colour through a mask 70 -> 43 and two with a
// gradient through another above it 117 -> 48.  What is left there: the vector
// instructions of the composite, and at 4 waves per SIMD the latency of the
// header, list and source loads.  Streaming stores took 3 to 6 % off.
enum BoxClass { kBoxSolid, kBoxGeneral };

template<int kClass, bool kDither>
__device__ __forceinline__ void render_box(const FrameDev& f, const FrameScratch& s, uint32_t n) {
  constexpr int kRows = 4;
  const uint32_t slot = xcd_tile(blockIdx.x);
  if (slot >= n) return;
  // headers: the fast bands' groups first, then the solid ones, then the
  // general ones
  const uint32_t n_fast = s.fgroup_off[f.n_bands], n_solid = s.sgroup_off[f.n_bands];
  if (slot >= (kClass == kBoxSolid ? n_solid : s.ggroup_off[f.n_bands])) return;
  if (s.flags && *s.flags) return;   // pool overflow: nothing is composited
  const uint32_t before = kClass == kBoxSolid ? n_fast : n_fast + n_solid;
  const pipe::CPtr<uint32_t> h = pipe::cptr((const uint32_t*)(s.group_hdr + 2 * ((size_t)before + slot)));
  const uint32_t lb = h[1], le = h[2], where = h[3], shape = h[7];
  const uint64_t ptr = ((uint64_t)h[5] << 32) | h[4];
  const int64_t stride = (int32_t)h[6];
  const int lane = threadIdx.x & 63;
  const int row0 = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)) * kRows;
  const int rows = min((int)((shape >> 16) & 0x1Fu) - row0, kRows);   // the wave's rows inside the canvas
  if (rows <= 0) return;
  const uint32_t tc0 = (where & 0xFFFFu) * kGroupTiles;
  const int X0 = (int)tc0 * kTileW, w = X0 + (int)(shape & 0xFFFFu);
  const int Y = (int)(where >> 16) * kTileH + row0;
  const bool a8 = (shape >> 21) & 1u;
  const bool fresh = (shape >> 22) & 1u;
  const int px = X0 + lane * 4;
  const int xr = min(X0 + (int)kGroupTiles * kTileW, w);   // right end of the group's pixels
  // the wave's first row, so that pixel x is at base + x * bytes per pixel
  uint8_t* const base = (uint8_t*)ptr + row0 * stride - (int64_t)X0 * (a8 ? 1 : 4);
  // masks of four pixels in a word
  const int n_in = min(max(w - px, 0), 4);
  const uint32_t in_mask = n_in == 4 ? 0xFFFFFFFFu : (1u << (8 * n_in)) - 1u;
  auto count = [&](uint32_t pm) {
    uint32_t c = 0;
#pragma unroll
    for (int k = 0; k < 4; k++) c += (uint32_t)__popcll(__ballot((pm & in_mask & (0xFFu << (8 * k))) != 0u));
    return c;
  };

  pipe::Px d[kRows][4];
#pragma unroll
  for (int r = 0; r < kRows; r++) {
#pragma unroll
    for (int k = 0; k < 4; k++) d[r][k] = pipe::px_of(0u);
    if (!fresh && r < rows) load_px<4>(base + r * stride, px, w, a8, d[r]);
  }
  // While the pixels of a fresh group are one value, that value alone is
  // composited.
  bool one = fresh && !a8;
  pipe::Px value[1] = {pipe::px_of(0u)};
  auto spread = [&]() {
    if (!one) return;
    one = false;
#pragma unroll
    for (int r = 0; r < kRows; r++)
#pragma unroll
      for (int k = 0; k < 4; k++) d[r][k] = value[0];
  };

  uint32_t npix = 0, touched = 0;   // touched: bit r, row r
  for (uint32_t chunk = lb; chunk < le; chunk += 64u) {
    // up to 64 commands in the lanes
    const uint32_t li = chunk + (uint32_t)lane;
    uint4 ent = make_uint4(0u, 0u, 0u, 0u);
    uint32_t style = 0;
    bool on = false;
    if (li < le) {
      ent = s.list_ent[li];
      style = s.list_style[li];
      on = (int)(ent.y & 0xFFFFu) < xr && (int)(ent.y >> 16) > X0 && (int)((ent.w >> kMetaRow0) & 31u) < row0 + rows &&
           (int)((ent.w >> kMetaRow1) & 31u) > row0;
    }
    for (uint64_t bits = __ballot(on); bits; bits &= bits - 1ull) {
      const uint32_t p = (uint32_t)__builtin_ctzll(bits);
      const uint32_t cmd = lane_value(ent.x, p), xs = lane_value(ent.y, p), meta = lane_value(ent.w, p), st = lane_value(style, p);
      const uint32_t alpha = (meta >> kMetaAlpha) & 0xFFu, op = (meta >> kMetaOp) & 7u, fetch = (meta >> kMetaFetch) & 7u;
      const int x0 = (int)(xs & 0xFFFFu), x1 = (int)(xs >> 16);
      const int ra = max((int)((meta >> kMetaRow0) & 31u) - row0, 0);
      const int rb = min((int)((meta >> kMetaRow1) & 31u) - row0, rows);   // rows ra .. rb - 1 (not empty)
      const uint32_t row_bits = (1u << rb) - (1u << ra);

      uint32_t pm[kRows];
      bool full = false;   // one mask, alpha, for every pixel of the group
      if ((meta & 3u) == kCmdBoxA) {
        // a box that goes past the canvas's right edge of the group takes
        // every lane: those pixels are neither counted nor stored, and a whole
        // wave under one mask is cheaper
        full = x0 <= X0 && x1 >= xr;
        uint32_t on4 = 0xFFFFFFFFu;
        if (!full) {
          const int n0 = min(max(x0 - px, 0), 4), n1 = min(max(x1 - px, 0), 4);
          on4 = (uint32_t)((1ull << (8 * n1)) - 1u) & ~(uint32_t)((1ull << (8 * n0)) - 1u);
        }
        pm[0] = on4 & (alpha * 0x01010101u);
        const uint32_t c = count(pm[0]);
        if (!c) continue;
        npix += c * (uint32_t)(rb - ra);
        touched |= row_bits;
        if (fetch == kFetchSolid && !a8 && op <= kOpSrcOver && full) {
          if (one && row_bits == (1u << rows) - 1u) {
            pipe::composite32_flat<1>(op, value, st, alpha);
            continue;
          }
          spread();
#pragma unroll
          for (int r = 0; r < kRows; r++)
            if ((row_bits >> r) & 1u) pipe::composite32_flat<4>(op, d[r], st, alpha);
          continue;
        }
#pragma unroll
        for (int r = 1; r < kRows; r++) pm[r] = pm[0];
      }
      else {
        box_mask_rows<kRows>(f, make_uint4(cmd, xs, 0u, meta), Y, px, pm);
        uint32_t any = 0;
#pragma unroll
        for (int r = 0; r < kRows; r++) {
          if (r >= rows) continue;
          const uint32_t c = count(pm[r]);
          npix += c;
          any |= (c ? 1u : 0u) << r;
        }
        if (!any) continue;
        touched |= any;
      }

      spread();
      // Sources that are colours or texels as they lie in memory: the four
      // rows together.
      const uint32_t fmt = (meta >> kMetaFmt) & 3u;
      if (!a8 && (fetch == kFetchSolid || (kClass == kBoxGeneral && pipe::fetches_rows(fetch, fmt)))) {
        uint32_t src[kRows][4];
#pragma unroll
        for (int r = 0; r < kRows; r++)
#pragma unroll
          for (int k = 0; k < 4; k++) src[r][k] = st;
        if (kClass == kBoxGeneral && fetch != kFetchSolid) {
          uint32_t any = pm[0];
#pragma unroll
          for (int r = 1; r < kRows; r++) any |= pm[r];
          if (any) pipe::fetch_rows<kRows>(pipe::cptr(f.styles + st), fetch, Y, px, f.images, fmt, src);
        }
#pragma unroll
        for (int r = 0; r < kRows; r++) {
          if (!((row_bits >> r) & 1u)) continue;
          pipe::Px sp[4];
#pragma unroll
          for (int k = 0; k < 4; k++) sp[k] = pipe::px_of(src[r][k]);
          if (kClass == kBoxGeneral && full && alpha == 255u && op == kOpSrcOver) {
            pipe::src_over_full<4>(d[r], sp, fetch != kFetchSolid);
            continue;
          }
          pipe::u16x2 mm[4];
#pragma unroll
          for (int k = 0; k < 4; k++) mm[k] = pipe::byte_pair(pm[r], k);
          pipe::composite32_n<4>(op, d[r], sp, mm, fetch != kFetchSolid);
        }
        continue;
      }
      // the rest a row at a time: the fetchers are long
#pragma unroll 1
      for (int r = ra; r < rb; r++) {
        pipe::Px t[4];
        uint32_t tp = 0;
#pragma unroll
        for (int q = 0; q < kRows; q++) {
          if (r != q) continue;
          tp = pm[q];
#pragma unroll
          for (int k = 0; k < 4; k++) t[k] = d[q][k];
        }
        uint32_t m[4];
#pragma unroll
        for (int k = 0; k < 4; k++) m[k] = (tp >> (8 * k)) & 0xFFu;
        apply_n<4, kDither>(f, s, meta, cmd, st, a8, 0u, Y + r, px, m, t);
#pragma unroll
        for (int q = 0; q < kRows; q++) {
          if (r != q) continue;
#pragma unroll
          for (int k = 0; k < 4; k++) d[q][k] = t[k];
        }
      }
    }
  }
  spread();
#pragma unroll
  for (int r = 0; r < kRows; r++)
    if ((touched >> r) & 1u) store_px<4, true>(base + r * stride, px, w, a8, d[r]);
  if (lane == 0) count_pixels(s, npix);
}

// Bands of solid SRC_OVER / SRC_COPY aligned boxes on 32-bit canvases, the pure
// compositing load, where nothing but loads in flight matters: pixels stay
// words (16 registers a lane) and are taken apart for one command at a time, so
// that eight waves fit a SIMD.  Ten 4K canvases with one SRC_OVER layer over
// what they hold: 116 us, 5.7 TB/s; 132 with the pixels as pairs throughout
// (five waves), 123 with records in LDS.  Four 4K canvases of three translucent
// layers over an opaque first fill: 31 us against 41 and 73.
__global__ __launch_bounds__(kTileThreads, 8) void k_render_box_fast(FrameDev f, FrameScratch s, uint32_t n) {
  constexpr int kRows = 4;
  const uint32_t slot = xcd_tile(blockIdx.x);
  if (slot >= n) return;
  // n is at most the number of all groups: the header, the first in the buffer,
  // is loaded together with the count and the pool flag
  const uint32_t n_groups = s.fgroup_off[f.n_bands], failed = s.flags ? *s.flags : 0u;
  const pipe::CPtr<uint32_t> h = pipe::cptr((const uint32_t*)(s.group_hdr + 2 * (size_t)slot));
  const uint32_t lb = h[1], le = h[2], where = h[3], shape = h[7];
  const uint64_t ptr = ((uint64_t)h[5] << 32) | h[4];
  const int64_t stride = (int32_t)h[6];
  if (slot >= n_groups || failed) return;
  const int lane = threadIdx.x & 63;
  const int row0 = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)) * kRows;
  const int rows = min((int)((shape >> 16) & 0x1Fu) - row0, kRows);   // the wave's rows inside the canvas
  if (rows <= 0) return;
  const int X0 = (int)((where & 0xFFFFu) * kGroupTiles) * kTileW, w = X0 + (int)(shape & 0xFFFFu);
  const int px = X0 + lane * 4;
  const int xr = min(X0 + (int)kGroupTiles * kTileW, w);   // right end of the group's pixels
  uint8_t* const base = (uint8_t*)ptr + row0 * stride - (int64_t)X0 * 4;
  const bool fresh = (shape >> 22) & 1u;

  uint32_t d[kRows][4];
#pragma unroll
  for (int r = 0; r < kRows; r++) {
#pragma unroll
    for (int k = 0; k < 4; k++) d[r][k] = 0u;
    if (!fresh && r < rows) load_words<4>(base + r * stride, px, w, d[r]);
  }
  // While the pixels of a fresh group are one value, that value alone is
  // composited.
  bool one = fresh;
  uint32_t value = 0u;
  auto spread = [&]() {
    if (!one) return;
    one = false;
#pragma unroll
    for (int r = 0; r < kRows; r++)
#pragma unroll
      for (int k = 0; k < 4; k++) d[r][k] = value;
  };

  uint32_t npix = 0, touched = 0;   // touched: bit r, row r
  for (uint32_t chunk = lb; chunk < le; chunk += 64u) {
    // up to 64 commands in the lanes
    const uint32_t li = chunk + (uint32_t)lane;
    uint32_t box_x = 0, box_meta = 0, style = 0;
    bool on = false;
    if (li < le) {
      const uint4 ent = s.list_ent[li];
      box_x = ent.y;
      box_meta = ent.w;
      style = s.list_style[li];
      on = (int)(box_x & 0xFFFFu) < xr && (int)(box_x >> 16) > X0 && (int)((box_meta >> kMetaRow0) & 31u) < row0 + rows &&
           (int)((box_meta >> kMetaRow1) & 31u) > row0 && ((box_meta >> kMetaAlpha) & 0xFFu);
    }
    for (uint64_t bits = __ballot(on); bits; bits &= bits - 1ull) {
      const uint32_t p = (uint32_t)__builtin_ctzll(bits);
      const uint32_t xs = lane_value(box_x, p), meta = lane_value(box_meta, p), color = lane_value(style, p);
      const uint32_t alpha = (meta >> kMetaAlpha) & 0xFFu, op = (meta >> kMetaOp) & 7u;
      const int x0 = (int)(xs & 0xFFFFu), x1 = (int)(xs >> 16);
      const int ra = max((int)((meta >> kMetaRow0) & 31u) - row0, 0);
      const int rb = min((int)((meta >> kMetaRow1) & 31u) - row0, rows);   // rows ra .. rb - 1 (not empty)
      const uint32_t row_bits = (1u << rb) - (1u << ra);
      touched |= row_bits;
      npix += (uint32_t)((min(x1, xr) - max(x0, X0)) * (rb - ra));
      const bool full = x0 <= X0 && x1 >= xr;
      if (one && full && row_bits == (1u << rows) - 1u) {
        pipe::Px v[1] = {pipe::px_of(value)};
        pipe::composite32_flat<1>(op, v, color, alpha);
        value = pipe::px_bits(v[0]);
        continue;
      }
      spread();
      // a box over the whole group takes every lane: pixels right of the canvas
      // aren't stored
      bool in[4];
#pragma unroll
      for (int k = 0; k < 4; k++) in[k] = full || (px + k >= x0 && px + k < x1);
#pragma unroll
      for (int r = 0; r < kRows; r++) {
        if (!((row_bits >> r) & 1u)) continue;
        pipe::Px v[4];
#pragma unroll
        for (int k = 0; k < 4; k++) v[k] = pipe::px_of(d[r][k]);
        pipe::composite32_flat<4>(op, v, color, alpha);
#pragma unroll
        for (int k = 0; k < 4; k++) d[r][k] = in[k] ? pipe::px_bits(v[k]) : d[r][k];
      }
    }
  }
  spread();
#pragma unroll
  for (int r = 0; r < kRows; r++)
    if ((touched >> r) & 1u) store_words<4, true>(base + r * stride, px, w, d[r]);
  if (lane == 0) count_pixels(s, npix);
}

__global__ __launch_bounds__(kTileThreads, 3) void k_render_box_solid(FrameDev f, FrameScratch s, uint32_t n) {
  render_box<kBoxSolid, false>(f, s, n);
}

template<bool kDither>
__global__ __launch_bounds__(kTileThreads, 4) void k_render_box(FrameDev f, FrameScratch s, uint32_t n) {
  render_box<kBoxGeneral, kDither>(f, s, n);
}

void launch_render(const FrameDev& f, const FrameScratch& s, uint32_t n_a, uint32_t strips, uint32_t n_f, uint32_t n_s, uint32_t n_g,
                   hipStream_t st) {
  if (!f.n_tiles) return;
  // frames with dithered gradients take the instances that carry the dither
  // path; the others leave it out
  if (n_a) {
    const dim3 grid = xcd_grid(n_a * strips), block(kTileThreads);
    if (strips == 4) {
      if (f.dither) hipLaunchKernelGGL((k_render<1, true>), grid, block, 0, st, f, s, n_a);
      else hipLaunchKernelGGL((k_render<1, false>), grid, block, 0, st, f, s, n_a);
    }
    else if (strips == 2) {
      if (f.dither) hipLaunchKernelGGL((k_render<2, true>), grid, block, 0, st, f, s, n_a);
      else hipLaunchKernelGGL((k_render<2, false>), grid, block, 0, st, f, s, n_a);
    }
    else if (f.dither) hipLaunchKernelGGL((k_render<4, true>), grid, block, 0, st, f, s, n_a);
    else hipLaunchKernelGGL((k_render<4, false>), grid, block, 0, st, f, s, n_a);
  }
  if (n_f) hipLaunchKernelGGL(k_render_box_fast, xcd_grid(n_f), dim3(kTileThreads), 0, st, f, s, n_f);
  if (n_s) hipLaunchKernelGGL(k_render_box_solid, xcd_grid(n_s), dim3(kTileThreads), 0, st, f, s, n_s);
  if (n_g && f.dither) hipLaunchKernelGGL(k_render_box<true>, xcd_grid(n_g), dim3(kTileThreads), 0, st, f, s, n_g);
  else if (n_g) hipLaunchKernelGGL(k_render_box<false>, xcd_grid(n_g), dim3(kTileThreads), 0, st, f, s, n_g);
}

void launch_tile_features(const FrameDev& f, const FrameScratch& s, uint32_t n_a, hipStream_t st) {
  if (!f.n_tiles || !n_a) return;
  hipLaunchKernelGGL(k_tile_features, dim3((n_a + 3) / 4), dim3(256), 0, st, f, s, n_a);
}

void launch_tile_queue(const FrameDev& f, const FrameScratch& s, uint32_t n_a, const float* pred, hipStream_t st) {
  if (!f.n_tiles || !n_a) return;
  launch_fill_u32(s.queue_hist, 0u, kQueueBuckets, st);
  hipLaunchKernelGGL(k_tile_keys, dim3((n_a + kQueueBuckets - 1) / kQueueBuckets), dim3(kQueueBuckets), 0, st, f, s, n_a, pred);
  hipLaunchKernelGGL(k_queue_scan, dim3(1), dim3(kQueueBuckets), 0, st, s);
  hipLaunchKernelGGL(k_tile_scatter, dim3((n_a + kQueueBuckets - 1) / kQueueBuckets), dim3(kQueueBuckets), 0, st, f, s, n_a);
}

void launch_render_queue(const FrameDev& f, const FrameScratch& s, uint32_t grid, uint32_t wgs_per_cu, hipStream_t st) {
  if (!f.n_tiles || !grid) return;
  if (!s.queue) launch_fill_u32(s.queue_head, 0u, 1, st);
  // Four workgroups per CU need the four-occupancy instance (128 VGPRs,
  // some spilled); fewer take the three-occupancy one (170 VGPRs).
  if (f.dither) {
    if (s.tile_cycles) hipLaunchKernelGGL((k_render_queue<true, 4, true>), dim3(grid), dim3(kTileThreads), 0, st, f, s);
    else if (wgs_per_cu >= 4) hipLaunchKernelGGL((k_render_queue<false, 4, true>), dim3(grid), dim3(kTileThreads), 0, st, f, s);
    else hipLaunchKernelGGL((k_render_queue<false, 3, true>), dim3(grid), dim3(kTileThreads), 0, st, f, s);
  }
  else if (s.tile_cycles) hipLaunchKernelGGL((k_render_queue<true, 4, false>), dim3(grid), dim3(kTileThreads), 0, st, f, s);
  else if (wgs_per_cu >= 4) hipLaunchKernelGGL((k_render_queue<false, 4, false>), dim3(grid), dim3(kTileThreads), 0, st, f, s);
  else hipLaunchKernelGGL((k_render_queue<false, 3, false>), dim3(grid), dim3(kTileThreads), 0, st, f, s);
}

}  // namespace b2amd
