// Drives the host side of a frame (blend2d_amd/csrc/context.cpp, compiled here
// with g++) on a stand-in device: HIP calls and kernel launches are replaced by
// functions below that keep account of device memory, the last error and the
// current device, and report the counts that a case asks for.  Nothing is
// rendered; what is checked is how often the edges run, with what buffers, and
// what the caller is told.
//
//   host_frame_check <case>      exit status 0 when the case holds
#include "../../blend2d_amd/csrc/context.cpp"

#include <stdlib.h>
#include <sys/mman.h>

#include <map>
#include <string>

namespace {

// ---- the stand-in device
size_t g_room = ~(size_t)0, g_used = 0;
std::map<void*, size_t> g_live;
hipError_t g_last = hipSuccess;
int g_device = 0;
struct Handle { int device; };

hipError_t fail(hipError_t e) { return g_last = e; }

// What the frame's edges need: segments of k_edges and of its clip list, and
// clip items, per region; from edge pass `later_from` on `later` more segments.
uint32_t g_segs = 0, g_clip_segs = 0, g_clip = 0, g_later = 0;
int g_later_from = 1 << 30;
// Edge passes so far, with their strides.
struct Pass { uint32_t seg_stride, clip_stride; };
std::vector<Pass> g_passes;
FrameScratch g_s{};
// Analytic tiles and binned segments that the scans report (0: no tiles, every
// segment in one band), and how the tiles were launched.
uint32_t g_tiles = 0, g_binned = 0, g_strips = 0;
bool g_queue = false;

uint32_t region_segs() {
  return g_segs + (g_clip <= g_s.clip_stride ? g_clip_segs : 0u) + ((int)g_passes.size() >= g_later_from ? g_later : 0u);
}

}  // namespace

extern "C" {
hipError_t hipMalloc(void** p, size_t n) {
  if (n > g_room - g_used) return fail(hipErrorOutOfMemory);
  *p = mmap(nullptr, n, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
  if (*p == MAP_FAILED) abort();
  g_live[*p] = n;
  g_used += n;
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  const auto it = g_live.find(p);
  if (it == g_live.end()) abort();
  g_used -= it->second;
  munmap(p, it->second);
  g_live.erase(it);
  return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { *p = calloc(1, n); return hipSuccess; }
hipError_t hipHostFree(void* p) { free(p); return hipSuccess; }
hipError_t hipGetLastError(void) { const hipError_t e = g_last; g_last = hipSuccess; return e; }
const char* hipGetErrorString(hipError_t) { return "stand-in error"; }
hipError_t hipGetDevice(int* d) { *d = g_device; return hipSuccess; }
hipError_t hipGetDeviceCount(int* n) { *n = 2; return hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { *v = 256; return hipSuccess; }
hipError_t hipDeviceSynchronize(void) { return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { *s = (hipStream_t) new Handle{g_device}; return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return fail(hipErrorNotSupported); }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t*) { return fail(hipErrorNotSupported); }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t*, hipGraph_t, hipGraphNode_t*, char*, size_t) { return fail(hipErrorNotSupported); }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return fail(hipErrorNotSupported); }
hipError_t hipEventCreate(hipEvent_t* e) { *e = (hipEvent_t) new Handle{g_device}; return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
// An event and the stream it is recorded in belong to one device.
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  return ((Handle*)e)->device == (s ? ((Handle*)s)->device : g_device) ? hipSuccess : fail(hipErrorInvalidHandle);
}
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { *ms = 0.f; return hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) { memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemcpy2D(void* d, size_t dp, const void* s, size_t sp, size_t w, size_t h, hipMemcpyKind) {
  for (size_t y = 0; y < h; y++) memcpy((char*)d + y * dp, (const char*)s + y * sp, w);
  return hipSuccess;
}
// (large canvases stay untouched: fresh mappings are zero)
hipError_t hipMemset(void* p, int v, size_t n) { if (v || n <= 1u << 20) memset(p, v, n); return hipSuccess; }
hipError_t hipMemsetD32(hipDeviceptr_t p, int v, size_t n) { for (size_t i = 0; i < n; i++) ((int*)p)[i] = v; return hipSuccess; }
}

namespace b2amd {
size_t scan_tmp_words(void) { return 16; }
EdgePlan edge_plan(uint32_t n_src) { return EdgePlan{8, 1, n_src >= 8192 ? kSegRegions : 1u}; }
void launch_frame_init(const FrameDev&, const FrameScratch&, hipStream_t) {}
void launch_edges(const FrameDev&, const FrameScratch& s, hipStream_t) {
  g_s = s;
  g_passes.push_back(Pass{s.seg_stride, s.clip_stride});
  // the buffers hold what their strides promise
  if (s.seg_stride) {
    const size_t slots = (size_t)s.seg_stride * s.seg_regions;
    const auto seg = g_live.find(s.segs), cmd = g_live.find(s.seg_cmd);
    if (seg == g_live.end() || seg->second < slots * sizeof(DevSeg)) abort();
    if (cmd == g_live.end() || cmd->second < ((size_t)(s.seg_rank - s.seg_cmd) + slots) * 4 || s.seg_rank < s.seg_cmd + slots) abort();
  }
  if (s.clip_stride) {
    const auto clip = g_live.find(s.clip);
    if (clip == g_live.end() || clip->second < (size_t)s.clip_stride * s.seg_regions * sizeof(ClipItem)) abort();
  }
}
void launch_report(const FrameScratch& s, uint32_t* report, hipStream_t) {
  memset(report, 0, kReportWords * 4);
  const uint32_t n = region_segs();
  for (uint32_t r = 0; r < s.seg_regions; r++) {
    report[kReportCursors + r] = n;
    report[kReportClip + r] = g_clip;
  }
  report[kCounterBinned] = g_tiles ? g_binned : n * s.seg_regions;
  report[kCounterTiles] = g_tiles;
  report[kCounterList] = 1;
}
void launch_bin_count(const FrameDev&, const FrameScratch&, uint64_t, hipStream_t) {}
void launch_scans(const FrameDev&, const FrameScratch&, hipStream_t) {}
void launch_setup(const FrameDev&, const FrameScratch&, hipStream_t) {}
void launch_bin_scatter(const FrameDev&, const FrameScratch&, uint64_t, hipStream_t) {}
void launch_render(const FrameDev&, const FrameScratch&, uint32_t n_a, uint32_t strips, uint32_t, uint32_t, uint32_t, hipStream_t) {
  if (n_a) g_strips = strips;
}
void launch_tile_features(const FrameDev&, const FrameScratch&, uint32_t, hipStream_t) {}
void launch_tile_queue(const FrameDev&, const FrameScratch&, uint32_t, const float*, hipStream_t) {}
void launch_render_queue(const FrameDev&, const FrameScratch&, uint32_t, uint32_t, hipStream_t) { g_queue = true; }
void launch_fill_u32(uint32_t*, uint32_t, size_t, hipStream_t) {}
void launch_gradient_luts(const lut::Job*, const lut::Stop*, uint32_t, uint32_t*, hipStream_t) {}
hipError_t noalloc_scratch(int, void**, size_t*) { return hipErrorNotSupported; }
namespace cm {
void launch_features(const FrameDev&, const FrameModel&, hipStream_t) {}
void launch_infer_frame(const FrameDev&, const FrameModel&, hipStream_t) {}
void launch_actuals(const FrameDev&, const FrameScratch&, const FrameModel&, uint32_t, hipStream_t) {}
void launch_mlp_forward(const float*, uint32_t, const float*, float*, hipStream_t) {}
uint32_t mlp_groups(uint32_t) { return 1; }
void launch_mlp_grad(const float*, const float*, uint32_t, const float*, float*, hipStream_t) {}
void launch_mlp_reduce(const float*, uint32_t, uint32_t, float*, hipStream_t) {}
void launch_adam(float*, const float*, float*, float*, uint32_t, float, hipStream_t) {}
}  // namespace cm
}  // namespace b2amd

namespace {

#define EXPECT(x) do { if (!(x)) { fprintf(stderr, "line %d: %s\n", __LINE__, #x); exit(1); } } while (0)

constexpr uint32_t kLines = 200000;   // sixteen regions of 12 500

struct Frame {
  BLAmdImage* img = nullptr;
  BLAmdContext* ctx = nullptr;
  explicit Frame(int w = 640, int h = 480) {
    EXPECT(bl_amd_image_create(&img, w, h, BL_AMD_FORMAT_PRGB32) == 0);
    EXPECT(bl_amd_context_create(&ctx) == 0);
    EXPECT(bl_amd_context_begin(ctx, img) == 0);
  }
  ~Frame() {
    bl_amd_context_destroy(ctx);
    bl_amd_image_destroy(img);
  }
  uint32_t flush() {
    std::vector<double> xy(2 * kLines);
    for (uint32_t i = 0; i < kLines; i++) { xy[2 * i] = (i * 37) % 640; xy[2 * i + 1] = (i * 101) % 480; }
    EXPECT(bl_amd_context_fill_polygon_d(ctx, xy.data(), kLines) == 0);
    g_passes.clear();
    return bl_amd_context_flush(ctx, 0);
  }
  Runner& runner() { return ctx->runner; }
};

void set_needs(uint32_t segs, uint32_t clip_segs, uint32_t clip) { g_segs = segs; g_clip_segs = clip_segs; g_clip = clip; }

// The guess holds the frame: one pass.
void enough() {
  Frame fr;
  set_needs(12000, 500, 400);
  EXPECT(fr.flush() == 0);
  EXPECT(g_passes.size() == 1);
}

// More segments than the guess: counted, then built; a third frame of the same
// size fits at once.
void more_segments() {
  Frame fr;
  set_needs(90000, 500, 400);
  EXPECT(fr.flush() == 0);
  EXPECT(g_passes.size() == 2 && g_passes[1].seg_stride >= 90500 && g_passes[1].clip_stride >= 400);
  EXPECT(fr.flush() == 0);
  EXPECT(g_passes.size() == 1);
}

// More clip items than the list: their segments are counted in a second pass.
void more_clip_items() {
  Frame fr;
  set_needs(12000, 1000, 12000);
  EXPECT(fr.flush() == 0);
  EXPECT(g_passes.size() == 2 && g_passes[1].clip_stride >= 12000);
  set_needs(12000, 200000, 30000);
  EXPECT(fr.flush() == 0);
  EXPECT(g_passes.size() == 3 && g_passes[2].clip_stride >= 30000 && g_passes[2].seg_stride >= 212000);
}

// A device without room for the guess, but for what the frame needs.
void tight_device() {
  size_t others;
  set_needs(12000, 500, 400);
  {
    Frame fr;
    EXPECT(fr.flush() == 0);
    const Runner& r = fr.runner();
    others = g_used - r.segs.cap - r.seg_cmd.cap - r.clip.cap;
  }
  EXPECT(g_used == 0);
  Frame fr;
  const size_t exact = (size_t)12500 * 16 * 24 * 5 / 4 + (size_t)400 * 16 * sizeof(ClipItem) * 5 / 4;
  g_room = others + exact + 65536;
  EXPECT(fr.flush() == 0);
  EXPECT(g_passes.size() == 3 && g_passes[2].seg_stride >= 12500 && g_passes[2].clip_stride >= 400);
}

// No room for the frame: OUT_OF_MEMORY, and the next frame with room is not
// told of it.
void too_tight() {
  set_needs(12000, 500, 400);
  Frame fr;
  g_room = g_used + ((size_t)8 << 20);
  EXPECT(fr.flush() == BL_AMD_ERROR_OUT_OF_MEMORY);
  g_room = ~(size_t)0;
  EXPECT(fr.flush() == 0);
  EXPECT(g_passes.size() == 1);
}

// A second pass that needs more than the first one counted is an error.
void counts_differ() {
  Frame fr;
  set_needs(90000, 500, 400);
  g_later = 1;
  g_later_from = 2;
  EXPECT(fr.flush() == BL_AMD_ERROR_DEVICE);
}

// Images are read back whatever device is current.
void other_device() {
  for (int pass = 0; pass < 2; pass++)
    for (int dev = 0; dev < 2; dev++) {
      g_device = dev;
      BLAmdImage* img = nullptr;
      EXPECT(bl_amd_image_create(&img, 33, 21, BL_AMD_FORMAT_PRGB32) == 0);
      std::vector<uint32_t> in(33 * 21), out(33 * 21);
      for (size_t i = 0; i < in.size(); i++) in[i] = (uint32_t)(i * 2654435761u) + (uint32_t)dev;
      EXPECT(bl_amd_image_upload(img, in.data(), 33 * 4) == 0);
      EXPECT(bl_amd_image_download(img, out.data(), 33 * 4) == 0);
      EXPECT(in == out);
      bl_amd_image_destroy(img);
    }
}

// How a frame never tuned runs its analytic tiles, on 256 CUs.
void schedules() {
  const struct { int w, h; uint32_t tiles, per_tile, strips; } cases[] = {
    {640, 480, 1, 1000, 4},        {1024, 1024, 384, 1000, 4},   {1024, 1024, 385, 1000, 2},
    {1024, 1024, 768, 1000, 2},    {1024, 1024, 769, 1000, 0},   {1024, 1024, 769, 63, 1},
    {2048, 2048, 2048, 64, 0},     {2048, 2048, 2049, 255, 1},   {2048, 2048, 2049, 256, 0},
    {8192, 8192, 16384, 256, 0},   {8192, 8192, 16385, 4000, 1}, {512, 65535, 16385, 4000, 1},
    {256, 65535, 16384, 256, 0},
  };
  set_needs(12000, 0, 0);
  for (const auto& c : cases) {
    Frame fr(c.w, c.h);
    g_tiles = c.tiles;
    g_binned = c.tiles * c.per_tile;
    g_segs = g_binned / 16 / 20 + 1;
    g_strips = 0;
    g_queue = false;
    EXPECT(fr.flush() == 0);
    if (g_queue != (c.strips == 0) || g_strips != c.strips)
      fprintf(stderr, "%u tiles of %u segments: queue %d strips %u\n", c.tiles, c.per_tile, g_queue, g_strips);
    EXPECT(g_queue == (c.strips == 0) && g_strips == c.strips);
  }
  // two canvases of bands of four tiles
  Frame a(256, 65535), b(256, 65535);
  BLAmdBatch* batch = nullptr;
  EXPECT(bl_amd_batch_create(&batch) == 0 && bl_amd_batch_add(batch, a.ctx) == 0 && bl_amd_batch_add(batch, b.ctx) == 0);
  const double xy[6] = {1, 1, 200, 3, 100, 90};
  EXPECT(bl_amd_context_fill_polygon_d(a.ctx, xy, 3) == 0 && bl_amd_context_fill_polygon_d(b.ctx, xy, 3) == 0);
  g_tiles = 32000;
  g_binned = 256 * 32000;
  g_segs = 4000;
  g_queue = false;
  EXPECT(bl_amd_batch_flush(batch) == 0);
  EXPECT(g_queue);
  bl_amd_batch_destroy(batch);
}

}  // namespace

int main(int argc, char** argv) {
  const std::map<std::string, void (*)()> cases = {
    {"enough", enough},           {"more_segments", more_segments}, {"more_clip_items", more_clip_items},
    {"tight_device", tight_device}, {"too_tight", too_tight},       {"counts_differ", counts_differ},
    {"other_device", other_device}, {"schedules", schedules}};
  const auto it = argc > 1 ? cases.find(argv[1]) : cases.end();
  if (it == cases.end()) return 2;
  it->second();
  puts("ok");
  return 0;
}
