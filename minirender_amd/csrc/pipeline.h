// pipeline.h -- launchers of the rasterization kernels (kernels.hip).
#pragma once

#include <hip/hip_runtime.h>

#include "common.h"
#include "exact.h"

namespace mr {

// The setup of an item and its id.
struct alignas(16) SetupRec {
  TriSetup s;
  uint32_t id;
};
static_assert(sizeof(SetupRec) == 64, "one record per 64 bytes");

// Device buffers and sizes of one batch.
struct BatchArgs {
  BinItem* items;            // [nregions * kRegion] survivors, per wavefront
  uint32_t* region_count;    // [nregions] survivors of each wavefront
  // Direct items of each job, behind the checkpoints in the checkpoint
  // buffer's last quarter (their number: direct_length in kernels.hip).
  BinItem* direct;           // [njobs * direct_cap]
  uint32_t direct_cap;
  int64_t nregions;
  // [ntiles * kCtrStride64] per tile: (walk work << 32) | (tile, triangle)
  // pairs, where a pair's walk work is its bbox pixels in the tile + 4 per
  // row + 16 (for the group leader's pair, times the group size); in the next
  // word, (direct entries << 32) | the first one's place in the bin list
  unsigned long long* tile_count;
  uint32_t* tile_off;        // [ntiles] first place in the bin list
  uint32_t* tile_cursor;     // [ntiles * kCtrStride] scatter cursors
  uint32_t* tile_heavy;      // [ntiles] merge slot of a split tile, kNoSlot, or kEmptyTile
  uint4* tile_list;          // [ntiles] {tile, first bin entry, entries, 1 if its job
                             // has direct items} of the tiles rastered whole: from the
                             // start those with entries (counters[kListed]), from the end
                             // those with direct entries only (kDirectTilesListed)
  uint32_t* tile_done;       // [ntiles] finished parts of a split tile
  uint2* parts;              // [parts_cap] (tile, part) of split tiles
  uint32_t parts_cap;
  uint2* bins;               // [bins_cap] (triangle id, draw) grouped by tile
  uint64_t bins_cap;
  // Edge checkpoints: the edge values of each row of a triangle spanning
  // several tile columns where the row enters each of them after the first
  // (written by the row pre-pass, read by the raster and shading).
  // Checkpoint of (row, column k of 2^cs pixels) of a survivor id, with
  // .y = columns | cs << 16: ckpt[ckpt_base[id].x + row * columns + k], with
  // .x a signed offset (the entries of the first column are allocated, never
  // written); .y == 0: no checkpoints.
  int2* ckpt_base;           // [2 * total_tris]
  float2* ckpt;              // [ckpt_cap], kCkptSegs equal segments
  uint64_t ckpt_cap;
  unsigned long long* ckpt_ctr;  // [kCkptSegs * kCtrStride] segment fill counters
  // Row tasks of the row pre-pass, (item index << 32) | pixel row, in
  // segments of half as many as the checkpoints' (a task per row of an
  // item with checkpoints, each row holding two entries or more); the
  // small segments' counters ckpt_ctr count them in their high 24 bits.
  unsigned long long* ckpt_rows;
  unsigned long long* heavy_keys;  // [heavy_cap * tile pixels] merge buffers
  uint32_t heavy_cap;
  uint32_t frag_size;        // max (tile, triangle) pairs per raster work item
  uint32_t band_work;        // a tile with more walk work is rastered in row bands
  unsigned long long* counters;     // [kNumCounters]
  // The counters' copy in pinned host memory (device address), written by
  // the shading kernel's first workgroup once they are final; null: the
  // host copies them back itself.
  unsigned long long* host_counters;
  // Per-workgroup statistics (no shared counter: same-address atomics
  // serialize): [0, kStatSlots) clipped triangles per geometry workgroup,
  // [kStatSlots, 2 kStatSlots) binned triangles per bin workgroup.
  unsigned long long* block_stats;
  float4* vscr;               // [total_verts] {px, py, zv, ez} of each projected vertex
  int64_t total_verts;
  const int64_t* vg_begin;    // [nvgroups] first record of each vertex group
  const int32_t* vg_draw;     // [nvgroups] a draw of the group (mesh, modelview, job)
  int32_t nvgroups;
  const DrawDesc* draws;
  const int64_t* draw_begin;  // [ndraws] tri_begin of each draw
  int32_t ndraws;
  const JobDesc* jobs;
  const int32_t* job_tile_base;   // [njobs]
  const int32_t* job_shade_base;  // [njobs]
  // Job hints: entry i = {job of tile (resp. shading block) i * kHintSpan,
  // first tile (block) of the next job or INT32_MAX}.
  const int2* tile_hint;          // [ceil(ntiles / kHintSpan)]
  const int2* shade_hint;         // [ceil(shade_blocks / kHintSpan)]
  int32_t njobs;
  int64_t total_tris;
  int32_t ntiles;
  int32_t tile_w, tile_h;    // each 8, 16 or 32
  int32_t raster_threads;    // workgroup size of the tile raster
  int32_t scan_blocks;
  int32_t shade_blocks;
  int32_t num_cus;
  int32_t geom_blocks;       // resident geometry workgroups (<= kStatSlots)
  // Where the edge checkpoints are taken (launched stages; the persistent
  // kernel always takes them in its binning stage): 1, by the scan's launch
  // in workgroups beside the scan, with the row pre-pass at the end of the
  // binning kernel (a batch of at most kCkptScanRegions regions, whose items
  // that pass reads while the scan runs); 0, by the binning
  // kernel, which reads the items anyway, with the row pre-pass a launch of
  // its own.
  int32_t ckpt_in_scan;
  // Setups of the items of a small batch, by item slot (in the checkpoint
  // buffer, which such a batch does not use).
  SetupRec* recs;
  uint2* region_box;         // behind them: {first | last << 16} column, row of each
                             // region's items
  // The kernels of the batch (launched stages).  front: geometry transforms
  // the vertices itself (k_front) and needs the batch counters zero before.
  // small: front, and the tiles test the items themselves (k_small).
  int32_t front, small;
  int32_t small_bands;       // workgroups per tile of k_small, each a band of its rows
};

// The argument of a batch's first kernel: with nwords, the batch tables too.
constexpr int kInlineWords = 832;
struct TableArgs {
  BatchArgs a;
  uint32_t nwords;
  alignas(16) uint32_t words[kInlineWords];
};

// Batches of at most this many triangles run k_front: beyond, transforming
// each vertex once costs less than once per corner (vertex and geometry
// kernels together 16.3 -> 12.0 us at 120 k triangles, 35 -> 32.5 at 1 M, but
// 55 -> 61 at 2.1 M).  Meshes that no call before has brought into a cache gain
// the same: 1.5 GB of meshes in turn, us a call with two kernels and one, 72.9
// and 66.5 at 100 k triangles, 103.8 and 96.9 at 1 M, 115.5 and 109.5 at 1.4 M.
constexpr int64_t kFrontTris = 1500000;
// Small batches (k_front and k_small, whose tiles test every region of their
// job): what the two kernels do sooner than the general ones (us a call, small
// and general; 64 triangles a region).
constexpr int kSmallWidth = 1024;  // rows are walked from the bbox's left column
constexpr int kSmallTiles = 8192;
constexpr int64_t kSmallTests = 800000;  // (tile, region) pairs tested
// The work that makes the general kernels the sooner ones, in pairs tested: a
// region is also set up and drawn tile by tile, a tile is a workgroup whose
// latency counts once a few rounds of them run.  Fitted to 750 calls of 1 to 150
// grids of 300 to 40,000 triangles at 33 x 33 to 1000 x 800; in 16-pixel tiles
// (their pairs, regions and tiles): one grid at 1000 x 800 of 9,000 (444,000, 141,
// 3,150) 48 and 56; 2 frames at 120 x 90 of 9,000 37 and 44; 16 at 250 x 250 of 4,700
// (303,000, 1,184, 4,096) 69 and 66, 30 of them 98 and 86; 150 at 120 x 90 of 2,500
// (288,000, 6,000, 7,200) 128 and 100.  A 32-pixel tile holds four times the pixels
// and their items: 32 frames at 250 x 250 of 1,000 (32,000, 512, 2,048) 77 and 78, of
// 4,700 (152,000, 2,368, 2,048) 99 and 80; 8 at 120 x 90 of 9,000 48 and 59.  In
// 8-pixel tiles: a sphere of 4 k at 640 x 480 (298,000, 62, 4,800) 37 and 68, 64
// frames at 64 x 64 of 4,700 (303,000, 4,736, 4,096) 85 and 63.
struct SmallWork {
  int64_t region, tile, most;
};
constexpr SmallWork small_work(int tile) {
  if (tile >= 32) return {60, 75, 300000};
  return {tile >= 16 ? 400 : 550, 75, 1200000};
}
// Regions of one job (k_small lists them in LDS): grids at 320 x 240 of 469 take
// 42 and 47, of 938 48 and 47, of 2,000 56 and 47; spheres 35 and 53, 39 and 53,
// 40 and 50.  The one wavefront of an 8-pixel tile tests them by itself: grids at
// 120 x 90 of 74 regions take 44 and 44, of 282 51 and 41, of 625 54 and 41 (at
// 250 x 250 39 and 47, 57 and 47, 60 and 47).
constexpr int kSmallRegions = 1536;
constexpr int small_ordered_regions(int tile) { return tile <= 8 ? 192 : kSmallRegions; }
// Regions of a job with triangles in no spatial order: every tile meets them
// all, where it meets 1 in 10 of a grid's.  For small triangles the general
// kernels are the better ones from about 7,000 on, large ones cost these more
// (they bin or list each for every tile), the larger and the more of them: so
// regions count in full, for 7/12 or not at all by the size of their
// triangles relative to the region.  At 640 x 480, sizes of 0.03, 0.12 and 0.21:
// 6,000 triangles 54 and 50, 66 and 97, 82 and 135; 16,000 95 and 55, 132 and
// 176, 169 and 298; 32,000 of the middle size 232 and 218.  Of 0.12 at other
// sizes of frame, 8,000 and 16,000: 96 x 64 61 and 79, 96 and 97; 320 x 240 73 and
// 76, 120 and 87; 1000 x 700 153 and 136, 265 and 217.
// Large ones count neither in small_work nor for small_ordered_regions (8,000 at
// 640 x 480 in 8-pixel tiles 884 and 3,239).
constexpr int64_t kSmallLoose = 112;
constexpr int32_t kScatterWeight = 12, kScatterMiddleWeight = 7;
constexpr double kScatterMiddle = 0.09, kScatterLarge = 0.16;
// A tile is drawn by one workgroup, or by up to 8, each a band of its rows,
// while that makes at most kSmallGroups (about what the GPU holds at once): a
// frame of few tiles left most CUs idle while each tile drew thousands of
// entries (4,000 overlapping triangles at 96 x 64 942 -> 160 us, 5,000 random
// ones 127 -> 60).  Frames of few regions gain nothing.
constexpr int kSmallGroups = 1024;
constexpr int64_t kSmallWholeRegions = 96, kSmallWholeLoose = 4;

constexpr int64_t kCkptScanRegions = 65536;

constexpr int kStatSlots = 8192;  // >= the geometry and bin grids

inline int32_t scan_blocks_for(int32_t tiles) {
  const int32_t per = kScanBlock * (tiles <= kScanWide ? 1 : kScanItems);
  return (tiles + per - 1) / per;
}

// Grid sizes of the grid-stride kernels (also used to sum their statistics).
// Workgroups of the geometry kernel, each taking one contiguous range of
// triangles: as many as the GPU holds at once (geom_blocks, from the
// kernel's occupancy), so none waits for a second round; a batch of more than
// 4096 triangles per such workgroup gets ~1024-triangle ranges instead, whose
// rounds even out the uneven draws of many jobs.
__host__ __device__ inline int32_t geom_grid(const BatchArgs& a) {
  const int64_t blocks = (a.total_tris + 255) / 256;
  int64_t g = a.geom_blocks;
  if (a.total_tris > g * 4096) {
    g = (a.total_tris + 1023) / 1024;
    if (g > kStatSlots) g = kStatSlots;
  }
  return (int32_t)(blocks < g ? blocks : g);
}
__host__ __device__ inline int32_t bin_grid(const BatchArgs& a) {
  // (At least a workgroup per 2048 pixels: the row pre-pass at the end has
  // many rows of few large triangles.)
  int64_t blocks = (a.nregions + 3) / 4;
  if (blocks < a.shade_blocks / 8) blocks = a.shade_blocks / 8;
  if (blocks < 1) blocks = 1;
  const int64_t cap = (int64_t)a.num_cus * 7;  // one resident round (7 per CU)
  return (int32_t)(blocks < cap ? blocks : cap);
}

// Workgroups that write the direct entries, 32 tiles a step each.
__host__ __device__ inline int32_t direct_grid(const BatchArgs& a) {
  if (a.direct_cap == 0) return 0;
  const int32_t steps = (a.ntiles + 31) / 32;
  return steps < 1024 ? steps : 1024;
}

// Copy the batch tables (TableLayout: a multiple of 16 bytes) from pinned host memory.
hipError_t launch_tables(const void* pinned, void* tables, size_t bytes, hipStream_t s);
hipError_t launch_clear(const BatchArgs& a, hipStream_t s);
hipError_t launch_vertex(const BatchArgs& a, hipStream_t s);
hipError_t launch_geometry(const BatchArgs& a, hipStream_t s);
// The batch's first kernel when a.front; tables (host memory) go inside its
// argument when they fit there, else they have been uploaded.
hipError_t launch_front(const BatchArgs& a, const void* tables, size_t table_bytes, hipStream_t s);
hipError_t launch_small(const BatchArgs& a, hipStream_t s);  // raster and shading when a.small
hipError_t launch_scan(const BatchArgs& a, hipStream_t s);
hipError_t launch_bin(const BatchArgs& a, hipStream_t s);
hipError_t launch_rows(const BatchArgs& a, hipStream_t s);  // nothing when ckpt_in_scan
hipError_t launch_tile(const BatchArgs& a, hipStream_t s);
// Geometry workgroups one CU holds at once (from the kernel's resources).
int geom_blocks_per_cu();
hipError_t launch_shade(const BatchArgs& a, hipStream_t s);
// The no-alloc entry point's scratch: kNoAllocScratchBytes of device memory
// per device (a static array).  noalloc_scratch_init(device), with that
// device current, looks up its address once (0, or -1 on failure);
// noalloc_scratch(device) returns it (null before the init).
constexpr size_t kNoAllocScratchBytes = (size_t)64 << 20;
constexpr int kMaxDevices = 64;
int noalloc_scratch_init(int device);
void* noalloc_scratch(int device);
// ---- the persistent kernel: every stage of a batch in one launch ----------
// Stages in queue order.
enum PersistStage : int32_t {
  kPClear, kPVertex, kPGeom, kPScan, kPBin, kPRows, kPTile, kPShade, kPStages
};
constexpr int kPQueues = 8;      // work queues (one per XCD under round-robin dispatch)
constexpr int kCtlStride = 32;   // u64 words between two control words (256 B)
// Control words (each kCtlStride words apart): queue heads and completed
// items per (stage, queue), queues completed per stage, completion flags per
// (stage, queue), workgroups finished, error.  Zero between launches: the
// last workgroup of a launch clears them.
constexpr int kCtlHead = 0;
constexpr int kCtlDone = kCtlHead + kPStages * kPQueues;
constexpr int kCtlFin = kCtlDone + kPStages * kPQueues;
constexpr int kCtlFlag = kCtlFin + kPStages;
constexpr int kCtlExit = kCtlFlag + kPStages * kPQueues;
constexpr int kCtlErr = kCtlExit + 1;
constexpr int kCtlWords = kCtlErr + 1;
constexpr size_t kCtlBytes = (size_t)kCtlWords * kCtlStride * 8;

struct PersistPlan {
  int32_t nvb[kPStages];    // workgroups of the stage's own launch (0: not run)
  int32_t depth[kPStages];  // items per workgroup a stage is dealt out in (>= 1)
  int32_t wait[kPStages];   // 1: the stage waits until every earlier stage is complete
  unsigned long long* ctl;  // kCtlBytes of control words, zero before the launch
  unsigned long long time_limit;  // wall-clock ticks one wait may take (0: every wait gives up)
  // Profiling (null: off): per stage s, words kStampStride * (2 s) and
  // kStampStride * (2 s + 1) take the maximum over workgroups of ~(first
  // wall-clock tick of the stage) and of its last tick; zero before the launch.
  unsigned long long* stamps;
};
constexpr int kStampStride = 32;
constexpr size_t kStampBytes = (size_t)2 * kPStages * kStampStride * 8;
// Launch the persistent kernel for a batch (16 x 16 tiles), on a grid of the
// workgroups the GPU holds at once.  `clear`: run the clear stage.
// wait_us: how long one wait may take, in microseconds (0: every wait gives
// up at once, which tests of the failure path use).
hipError_t launch_persistent(const BatchArgs& a, bool clear, unsigned long long* ctl,
                             unsigned long long* stamps, uint64_t wait_us, hipStream_t s);
// Wall-clock ticks per second of the device's clock (wall_clock64).
unsigned long long wall_clock_hz();
bool persistent_supported(int tile_w, int tile_h);

bool tile_supported(int tile_w, int tile_h);
// Raster workgroup sizes built per tile size: 8x8 {64, 128}, 16x16 and
// 32x32 {64, 128, 256, 512}; the default is 64 for 8x8, else 256.
bool raster_threads_supported(int tile_w, int threads);
int default_raster_threads(int tile_w);

}  // namespace mr
