// CPU check of the host side of a batch (context.cpp), built with g++ against
// the stand-ins below for the HIP runtime and for the kernel launchers: what
// is launched, counted and assumed of buffers from one call to the next.
//   clean     a general batch finds the tile counters zero, whatever ran and
//             grew the buffers before it
//   launches  mr_stats.launches is the number of kernels launched (replayed)
//   small     which batches the two kernels of small batches get, and in how
//             many row bands per tile
// Device memory is host memory, filled with 0xAB when it is allocated; a freed
// block's address is the next allocation's.  A general batch's launches
// check that the counters they add to are zero, and leave them so at the end,
// as the kernels do.  Prints "ok" or the first failure.
#include <sys/mman.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <string>
#include <vector>

#include "minirender_amd.h"
#include "pipeline.h"

#define FAIL(...) (printf(__VA_ARGS__), printf("\n"), exit(1))

// ---- the HIP runtime --------------------------------------------------------
static std::vector<void*> g_free;
static std::string* g_captured = nullptr;  // the graph being captured
static int g_updates = 0;
static void* block(size_t bytes) {
  constexpr size_t kBlock = (size_t)1 << 32;
  if (bytes > kBlock) return nullptr;
  void* p;
  if (!g_free.empty()) {
    p = g_free.back();
    g_free.pop_back();
  } else {
    p = mmap(nullptr, kBlock, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
    if (p == MAP_FAILED) return nullptr;
  }
  memset(p, 0xAB, bytes);
  return p;
}

extern "C" {
hipError_t hipMalloc(void** p, size_t n) { return (*p = block(n)) ? hipSuccess : hipErrorOutOfMemory; }
hipError_t hipFree(void* p) { if (p) g_free.push_back(p); return hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return hipMalloc(p, n); }
hipError_t hipHostFree(void* p) { return hipFree(p); }
hipError_t hipHostGetDevicePointer(void** d, void* h, unsigned) { *d = h; return hipSuccess; }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) { memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemset(void* d, int v, size_t n) { memset(d, v, n); return hipSuccess; }
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) { memset(d, v, n); return hipSuccess; }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void*) { a->type = hipMemoryTypeUnregistered; return hipSuccess; }
hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { *v = 256; return hipSuccess; }
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { *s = (hipStream_t)malloc(1); return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { free(s); return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
// A graph is the names of the kernels launched while it was captured; an update
// keeps the kernels, so it has to be of the same ones.
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { g_captured = new std::string; return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) { *g = (hipGraph_t)g_captured; g_captured = nullptr; return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t g) { delete (std::string*)g; return hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t g, hipGraphNode_t*, char*, size_t) { *e = (hipGraphExec_t)new std::string(*(std::string*)g); return hipSuccess; }
hipError_t hipGraphExecUpdate(hipGraphExec_t e, hipGraph_t g, hipGraphNode_t*, hipGraphExecUpdateResult* r) {
  if (*(std::string*)e != *(std::string*)g) FAIL("a graph of %s updated by one of %s", ((std::string*)e)->c_str(), ((std::string*)g)->c_str());
  g_updates++;
  *r = hipGraphExecUpdateSuccess;
  return hipSuccess;
}
hipError_t hipGraphExecDestroy(hipGraphExec_t e) { delete (std::string*)e; return hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { *e = (hipEvent_t)malloc(1); return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) { free(e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { *ms = 0; return hipSuccess; }
}

// ---- the launchers ----------------------------------------------------------
namespace mr {
static int g_launches = 0;  // kernels launched
static bool g_general = false, g_small = false;
static int g_bands = 0;  // of the last small batch

static void launched(const char* name, int kind = 0) {
  g_launches++;
  if (g_captured) *g_captured += name + std::to_string(kind) + " ";
}

static void zero(const BatchArgs& a) {
  memset(a.counters, 0, kNumCounters * 8);
  memset(a.ckpt_ctr, 0, (size_t)kCkptSegs * kCtrStride * 8);
}
static void zero_tiles(const BatchArgs& a) {
  for (int i = 0; i < a.ntiles; i++) {
    memset(a.tile_count + (size_t)i * kCtrStride64, 0, 6 * 8);
    a.tile_done[i] = 0;
  }
}
static void expect_zero(const BatchArgs& a) {
  for (int i = 0; i < kNumCounters; i++)
    if (a.counters[i]) FAIL("batch counter %d not zero", i);
  for (int i = 0; i < kCkptSegs; i++)
    if (a.ckpt_ctr[i * kCtrStride]) FAIL("checkpoint counter %d not zero", i);
  for (int i = 0; i < a.ntiles; i++)
    if (a.tile_count[(size_t)i * kCtrStride64] || a.tile_done[i]) FAIL("counters of tile %d of %d not zero", i, a.ntiles);
}
static void hand_counters(const BatchArgs& a) {
  if (!a.host_counters) return;
  memcpy(a.host_counters, a.counters, kNumCounters * 8);
  zero(a);
}

hipError_t launch_tables(const void* p, void* t, size_t n, hipStream_t) { launched("tables"); memcpy(t, p, n); return hipSuccess; }
hipError_t launch_clear(const BatchArgs& a, hipStream_t) { launched("clear"); zero(a); zero_tiles(a); return hipSuccess; }
hipError_t launch_vertex(const BatchArgs& a, hipStream_t) { if (a.total_verts) launched("vertex"), zero(a); return hipSuccess; }
static hipError_t geometry(const BatchArgs& a) {
  launched("geometry", 2 * a.front + a.small);
  g_general = !a.small;
  if (a.small) return hipSuccess;
  expect_zero(a);
  for (int i = 0; i < a.ntiles; i++) a.tile_count[(size_t)i * kCtrStride64] = 1, a.tile_done[i] = 1;
  return hipSuccess;
}
hipError_t launch_geometry(const BatchArgs& a, hipStream_t) { return a.total_tris ? geometry(a) : hipSuccess; }
hipError_t launch_front(const BatchArgs& a, const void*, size_t, hipStream_t) { return geometry(a); }
hipError_t launch_small(const BatchArgs& a, hipStream_t) {
  launched("small", 2 * a.tile_w + (a.small_bands > 1));
  g_small = true;
  g_bands = a.small_bands;
  if (a.small_bands < 1 || a.tile_h % a.small_bands || (a.small_bands > 1 && a.small_bands * a.ntiles > kSmallGroups))
    FAIL("%d bands of %d rows, %d tiles", a.small_bands, a.tile_h, a.ntiles);
  memset(a.host_counters, 0, kNumCounters * 8);
  return hipSuccess;
}
hipError_t launch_scan(const BatchArgs&, hipStream_t) { launched("scan"); return hipSuccess; }
hipError_t launch_bin(const BatchArgs& a, hipStream_t) { launched("bin", a.ckpt_in_scan); return hipSuccess; }
hipError_t launch_rows(const BatchArgs& a, hipStream_t) { if (!a.ckpt_in_scan) launched("rows"); return hipSuccess; }
hipError_t launch_tile(const BatchArgs& a, hipStream_t) { launched("tile", 2 * a.tile_w + few_tiles(a.ntiles)); return hipSuccess; }
hipError_t launch_shade(const BatchArgs& a, hipStream_t) { launched("shade"); zero_tiles(a); hand_counters(a); return hipSuccess; }
hipError_t launch_persistent(const BatchArgs& a, bool clear, unsigned long long*, unsigned long long*, uint64_t, hipStream_t) {
  launched("persistent");
  if (clear) zero_tiles(a);
  zero(a);
  expect_zero(a);
  return hipSuccess;
}
int geom_blocks_per_cu() { return 7; }
int noalloc_scratch_init(int) { return -1; }
void* noalloc_scratch(int) { return nullptr; }
unsigned long long wall_clock_hz() { return 100000000ull; }
bool persistent_supported(int w, int h) { return w == 16 && h == 16; }
bool tile_supported(int w, int h) { return w == h && (w == 8 || w == 16 || w == 32); }
bool raster_threads_supported(int, int) { return true; }
int default_raster_threads(int) { return 256; }
}  // namespace mr

// ---- calls ------------------------------------------------------------------
static mr_ctx* open_ctx() {
  mr_ctx* c;
  if (mr_ctx_create(0, 0, &c)) FAIL("context");
  return c;
}
// strip: neighbouring triangles share corners; else each has its own.
static int32_t upload(mr_ctx* c, int ntri, bool strip = false) {
  std::vector<float> v(9 * (size_t)ntri);
  std::vector<int32_t> ix(3 * (size_t)ntri);
  for (int i = 0; i < 3 * ntri; i++) ix[i] = strip ? i / 3 + i % 3 : i;
  int32_t h;
  if (mr_mesh_upload(c, v.data(), 3 * ntri, v.data(), 3 * ntri, nullptr, 0, ix.data(), ix.data(), nullptr, ntri, &h))
    FAIL("upload");
  return h;
}
// `n` frames of `ndraws` draws of a mesh, their images in host memory; returns
// the kernels launched.
static int render(mr_ctx* c, int32_t mesh, int ndraws, int w, int h, int n = 1) {
  std::vector<mr_draw> draws(ndraws);
  for (mr_draw& d : draws) {
    memset(&d, 0, sizeof(d));
    d.mesh = mesh;
    d.texture = -1;
  }
  mr_frame f;
  memset(&f, 0, sizeof(f));
  f.width = w;
  f.height = h;
  f.draws = draws.data();
  f.ndraws = ndraws;
  f.projection[15] = 1.0f;
  std::vector<uint8_t> rgb((size_t)3 * w * h);
  mr_outputs o;
  memset(&o, 0, sizeof(o));
  o.rgb8 = rgb.data();
  const std::vector<mr_frame> frames(n, f);
  const std::vector<mr_outputs> outs(n, o);
  const int before = mr::g_launches;
  mr::g_general = mr::g_small = false;
  const int rc = mr_render_batch(c, frames.data(), n, outs.data());
  if (rc) FAIL("%d x %d: status %d", w, h, rc);
  return mr::g_launches - before;
}

static void check_clean() {
  mr_ctx* c = open_ctx();
  const int32_t mesh = upload(c, 4);
  const int sizes[][2] = {{1100, 100}, {640, 480}, {1000, 700}, {1100, 100}, {1100, 700}, {1000, 1000}, {1100, 100},
                          {64, 64}, {1100, 1200}};
  for (auto& s : sizes) {
    render(c, mesh, 1, s[0], s[1]);
    if (mr::g_small != (s[0] <= 1024) || mr::g_general != (s[0] > 1024)) FAIL("%d x %d: route", s[0], s[1]);
  }
  mr_ctx_destroy(c);
}

static void check_launches() {
  mr_ctx* c = open_ctx();
  const int32_t mesh = upload(c, 4);
  // Tables inside the argument, copied, fetched by a kernel; small, general,
  // empty frames; the persistent kernel (one launch).
  const int draws[] = {1, 20, 60, 0}, widths[] = {300, 1100};
  for (int persistent = 0; persistent < 2; persistent++) {
    mr_ctx_set_persistent(c, persistent);
    for (int w : widths)
      for (int n : draws) {
        const int count = render(c, mesh, n, w, 200);
        mr_stats st;
        mr_ctx_get_stats(c, &st);
        if (st.launches != count || (persistent && count != 1))
          FAIL("%d draws, width %d, persistent %d: %d launches, counted %d", n, w, persistent, count, (int)st.launches);
      }
  }
  // Replays launch what was captured, whatever ran in between.
  mr_ctx_set_persistent(c, 0);
  mr_ctx_set_graphs(c, 1);
  int captured[2];
  for (int rep = 0; rep < 4; rep++)
    for (int k = 0; k < 2; k++) {
      const int count = render(c, mesh, 1, widths[k], 200);
      if (count) captured[k] = count;
      mr_stats st;
      mr_ctx_get_stats(c, &st);
      if (st.launches != captured[k] || (rep == 3 && count))
        FAIL("replay %d of width %d: counted %d of %d", rep, widths[k], (int)st.launches, captured[k]);
    }
  mr_ctx_destroy(c);
}

static void check_small() {
  mr_ctx* c = open_ctx();
  render(c, upload(c, 4), 1, 3840, 2160);  // buffers large enough for all below
  const struct { int ntri; bool strip; int w, h, n, bands; } cases[] = {
      {64, true, 96, 64, 1, 1},         // few regions
      {4000, true, 96, 64, 1, 1},
      {7000, true, 96, 64, 1, 8},       // 24 tiles
      {5000, false, 256, 128, 1, 8},    // 128 tiles
      {5000, false, 250, 145, 1, 4},    // 160 tiles
      {5000, false, 512, 256, 1, 2},
      {5000, false, 432, 304, 1, 1},    // 513 tiles
      {7168, false, 320, 240, 1, 2},    // 112 loose regions
      {7169, false, 320, 240, 1, 0},    // one more
      {20000, false, 640, 480, 1, 0},
      {20000, true, 640, 480, 1, 1},
      {98304, true, 320, 240, 1, 2},    // 1,536 regions
      {98305, true, 320, 240, 1, 0},
      {4713, true, 250, 250, 12, 1},    // 3,072 tiles
      {4713, true, 250, 250, 16, 1},    // 303,000 tests of 4,096 tiles
      {4713, true, 250, 250, 18, 0},
      {1500, true, 250, 250, 30, 1},
      {9024, true, 120, 90, 8, 2},      // 141 regions a job
      {9024, true, 120, 90, 24, 0},
  };
  for (auto& k : cases) {
    render(c, upload(c, k.ntri, k.strip), 1, k.w, k.h, k.n);
    if (mr::g_small != (k.bands != 0) || (k.bands && mr::g_bands != k.bands))
      FAIL("%d triangles (strip %d), %d of %d x %d: small %d, %d bands, not %d", k.ntri, k.strip, k.n, k.w, k.h,
           mr::g_small, mr::g_bands, k.bands);
  }
  mr_ctx_destroy(c);
}

// Loose triangles of side `side` with centres in a box of side 1; shared: the
// mesh refers to the vertices of another one.
static int32_t upload_loose(mr_ctx* c, int ntri, float side, bool shared) {
  std::vector<float> v(9 * (size_t)ntri);
  std::vector<int32_t> ix(3 * (size_t)ntri);
  unsigned seed = 1;
  auto rnd = [&] { return (float)((seed = seed * 1664525u + 1013904223u) >> 8) / 16777216.0f; };
  for (int t = 0; t < ntri; t++) {
    const float m[3] = {rnd(), rnd(), rnd()};
    for (int k = 0; k < 9; k++) v[9 * (size_t)t + k] = m[k % 3] + (k / 3 == k % 3 ? side : 0.0f);
  }
  for (int i = 0; i < 3 * ntri; i++) ix[i] = i;
  int32_t h, first[3] = {0, 1, 2};
  const int32_t* own = shared ? first : ix.data();
  if (mr_mesh_upload(c, v.data(), 3 * ntri, v.data(), 3 * ntri, nullptr, 0, own, own, nullptr, shared ? 1 : ntri, &h))
    FAIL("upload");
  if (shared && mr_mesh_upload_shared(c, h, ix.data(), ix.data(), nullptr, ntri, &h)) FAIL("shared upload");
  return h;
}

static void check_scatter() {
  mr_ctx* c = open_ctx();
  render(c, upload(c, 4), 1, 3840, 2160);  // buffers large enough for all below
  const struct { int ntri; float side; bool small; } cases[] = {
      {7168, 0.03f, true}, {7169, 0.03f, false},   // 112 regions of small triangles
      {12288, 0.14f, true}, {12353, 0.14f, false}, // 192 of middling ones (0.14 / 1.14 of the region)
      {8000, 0.3f, true}, {20000, 0.3f, true},     // large ones count by the other limits only
      {98304, 0.3f, true}, {98305, 0.3f, false},
  };
  for (auto& k : cases)
    for (int shared = 0; shared < 2; shared++) {
      render(c, upload_loose(c, k.ntri, k.side, shared), 1, 320, 240);
      if (mr::g_small != k.small) FAIL("%d triangles of %g, shared %d: small %d", k.ntri, k.side, shared, mr::g_small);
    }
  render(c, upload_loose(c, 5000, 0.3f, false), 2, 320, 240);
  if (!mr::g_small) FAIL("two draws");
  render(c, upload_loose(c, 5000, 0.03f, true), 2, 320, 240);
  if (mr::g_small) FAIL("two draws of small triangles");
  mr_ctx_destroy(c);
}

static void check_tiles() {
  mr_ctx* c = open_ctx();
  render(c, upload(c, 4), 1, 3840, 2160);  // buffers large enough for all below
  const struct { int tile, ntri, w, h, n; bool small; } cases[] = {
      {8, 12288, 120, 90, 1, true}, {8, 12289, 120, 90, 1, false},    // 192 regions
      {16, 12289, 120, 90, 1, true},
      {16, 2560, 120, 90, 54, true}, {16, 2560, 120, 90, 56, false},  // 40 regions, 48 tiles a frame
      {16, 9024, 1000, 800, 1, true},
      {32, 4736, 250, 250, 20, true}, {32, 4736, 250, 250, 22, false},  // 74 regions, 64 tiles
      {32, 1024, 250, 250, 40, true}, {32, 1024, 250, 250, 64, false},
      {32, 640, 250, 250, 64, false}, {32, 9024, 120, 90, 8, true},
      {8, 4736, 64, 64, 20, true}, {8, 4736, 64, 64, 32, false},
      {8, 3968, 640, 480, 1, true}, {8, 3968, 200, 150, 12, true},
  };
  for (auto& k : cases) {
    mr_ctx_set_tile(c, k.tile, k.tile);
    render(c, upload(c, k.ntri, true), 1, k.w, k.h, k.n);
    if (mr::g_small != k.small) FAIL("%d triangles, %d of %d x %d, tile %d: small %d", k.ntri, k.n, k.w, k.h, k.tile, mr::g_small);
  }
  mr_ctx_set_tile(c, 8, 8);
  for (int ntri : {20000, 8000}) {
    render(c, upload_loose(c, ntri, 0.3f, false), 1, ntri == 20000 ? 320 : 640, ntri == 20000 ? 240 : 480);
    if (!mr::g_small) FAIL("%d large loose triangles, tile 8", ntri);
  }
  mr_ctx_set_tile(c, 16, 16);
  render(c, upload_loose(c, 12000, 0.3f, true), 1, 1000, 1000);
  if (!mr::g_small) FAIL("large loose triangles, 3,969 tiles");
  mr_ctx_destroy(c);
}

// Frames of many sizes in turn, replayed: a graph is updated in place to one of
// the same kernels only.
static void check_graphs() {
  mr_ctx* c = open_ctx();
  mr_ctx_set_graphs(c, 1);
  const int32_t few = upload(c, 64, true), many = upload(c, 7000, true);
  const int sizes[][2] = {{96, 64}, {90, 60}, {250, 145}, {640, 480}, {600, 400}, {1000, 700}, {1100, 64}, {1100, 80}, {1100, 1000}, {1200, 900}};
  for (int rep = 0; rep < 3; rep++)
    for (int tile : {16, 32}) {
      mr_ctx_set_tile(c, tile, tile);
      for (auto& s : sizes) render(c, few, 1, s[0], s[1]);
      for (auto& s : sizes) render(c, many, 1, s[0], s[1]);
    }
  if (!g_updates) FAIL("no graph was updated");
  mr_ctx_destroy(c);
}

int main(int argc, char** argv) {
  const char* what = argc > 1 ? argv[1] : "";
  if (!strcmp(what, "clean")) check_clean();
  else if (!strcmp(what, "launches")) check_launches();
  else if (!strcmp(what, "small")) check_small();
  else if (!strcmp(what, "scatter")) check_scatter();
  else if (!strcmp(what, "tiles")) check_tiles();
  else if (!strcmp(what, "graphs")) check_graphs();
  else FAIL("nothing to check");
  printf("ok\n");
  return 0;
}
